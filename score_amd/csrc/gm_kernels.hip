/*
 * gm_kernels.hip -- gfx950 kernels of the growth machine.
 *
 * One growth step of SCORE (SCORE_Kernel.cpp:6635-6654 with OMP_NUM_THREADS=1)
 * is, in serial order: sweep the Inside list, sweep the Border list, let every
 * completed Inside cell infect its 26 neighbours in list order, then every
 * completed Border cell.  A target is won by the first attempt in that order
 * that finds it deformed.  Steps run in launch windows of up to GM_WMAX; the same
 * outcome is computed by
 *
 * per window
 *   k_reanchor     only where the scalars changed: every active cell is advanced to
 *                  the step with its old increment and predicted again with the new
 *                  one, one thread per slot.
 *   k_arrivals     only where nuclei arrive at the window's first step.
 *   k_sweep        pass over the completion codes of the occupied slots: per block,
 *                  the cells that complete in each step of the window and the
 *                  INACTIVE slots.
 *   k_sweep_scan   one block scans the per-block counts into offsets (short fronts:
 *                  each block of the next pass adds up what it needs).
 *   k_compact      the completed slots of every step in FullRX order (Inside list,
 *                  then Border), and the INACTIVE slots as masks.  Short fronts: the
 *                  first step's propose pass too.
 *   (k_window_end  closes the last step and hands the stats to the host, where the last
 *                  commit pass has not done it: a halted window)
 * per step
 *   k_propose      block 0 closes the step before (its row, list lengths, recycling
 *                  tables).  The others copy what the infection needs of each
 *                  completed cell (ids, rxFrac after the completing addition, P,
 *                  coordinates) into dense parent planes; every (parent p, direction
 *                  rank r) attempt on a deformed cell (one bit of a brick-blocked
 *                  bitmap) does atomicMin(claim[target], p*32 + r): the key orders
 *                  attempts exactly as the serial loop issues them.
 *   k_decide       an attempt wins iff its key is the minimum; winners per parent
 *                  and destination list as bit masks, counted per 64 parents and per
 *                  block; the parents retire.  Further blocks write the recycled
 *                  slots that may be handed out, ascending.
 *   k_commit       the winners before a block rank its own: rank k into a list takes
 *                  the k-th recycled slot, else appends.  One thread per winner writes
 *                  the new record with its increment and completion step (certified
 *                  from the real sums, gm_radd_count_to_one), and clears the cell's
 *                  bitmap bit.  The window's last one ends it (window_end).
 *
 * Three passes a step, where sweep, scan, compaction, ranking scan, recycling and
 * the step's row were seven more launches: on the 24x20x18 domain of ten nuclei a
 * step went from 48 to 20 us, at 100^3 from 62 to 26, at 320^3 from 90 to 54, at
 * 512^3 from 165 to 132.  A pass costs 2.4 us whatever it does and 0.7 us more for
 * every load that waits for another, so on fronts of a few thousand parents the length
 * of these chains and the number of passes are the time.
 *
 * No kernel waits on another block: every cross-block dependency is a kernel
 * boundary, but for the end of a window, which the last block to finish takes over,
 * so the passes use only relaxed device atomics.  FP64 throughout,
 * compiled with -ffp-contract=off so every product and sum is rounded exactly as
 * in the reference's build without FMA.
 */
#include "gm_device.h"

/* ---------------------------------------------------------------- helpers */

__global__ void k_fill_u32(uint32_t *p, uint32_t v, size_t n) {
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) p[i] = v;
}
__global__ void k_fill_u64(unsigned long long *p, unsigned long long v, size_t n) {
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) p[i] = v;
}

hipError_t gm_launch_fill_u32(uint32_t *p, uint32_t v, size_t n, hipStream_t s) {
    if (n == 0) return hipSuccess;
    k_fill_u32<<<fill_blocks(n), GM_BLOCK, 0, s>>>(p, v, n);
    return hipGetLastError();
}
hipError_t gm_launch_fill_u64(unsigned long long *p, unsigned long long v, size_t n, hipStream_t s) {
    if (n == 0) return hipSuccess;
    k_fill_u64<<<fill_blocks(n), GM_BLOCK, 0, s>>>(p, v, n);
    return hipGetLastError();
}

/* The per-step scalars changed: every active cell is advanced to the start of
 * step k with its old increment (its anchor moves to k) and predicted again
 * with the new one.  One thread per occupied slot.  Codes of cells that
 * completed before step k are turned into INACTIVE. */
__global__ void __launch_bounds__(GM_BLOCK) k_reanchor(GmDev d, GmSweepArgs A) {
    const uint32_t nI = d.st->nI, n = nI + d.st->nB;
    const uint32_t kc = A.k & (GM_CS_MOD - 1u);
    for (uint32_t i = blockIdx.x * GM_BLOCK + threadIdx.x; i < n; i += gridDim.x * GM_BLOCK) {
        const uint32_t s = occ_slot(d, nI, i);
        const uint32_t cs = d.cstep[s];
        if (cs_inactive(cs, kc, d.horizon)) {
            /* a cell that completed in an earlier step: its code becomes the sentinel */
            if (cs != GM_CS_INACTIVE) d.cstep[s] = (gm_cs_t)GM_CS_INACTIVE;
            continue;
        }
        GmRec *r = d.rec + s;
        const RecA a = rec_a(r);
        const RecC c = rec_c(r);
        double f = a.frac0;
        if (cs != GM_CS_UNKNOWN) {
            const double inc = r->inc;
            /* one step since the anchor: the one addition itself */
            f = A.k - a.s0 == 1u ? f + inc : gm_radd_n(f, inc, A.k - a.s0);
        }
        const double P = resolved(d, c.P);
        if (is_pending(c.P)) r->P = P;
        predict_slot(d, A, s, f, A.k, P, c.defg, a.inf);
    }
}

/* ------------------------------------------------------------ window sweep
 * A cell infected inside a launch window cannot complete before the window ends
 * (window_length, gm_host.cpp), so one pass over the completion codes at the
 * window's start finds the completed cells of all its steps: SCORE's sweep
 * (calcGrowthStepInside / Border, SCORE_Kernel.cpp:4046-4249) with its FullRX
 * lists, W steps at a time.  The 2-byte codes are read twice per window instead
 * of once per step.
 *
 * Blocks of GM_BLOCK threads own consecutive 512-slot chunks of one list, P.cpw
 * per wave: blocks [0, P.nbI) the Inside list, [P.nbI, P.nb) the Border list, so
 * block order is FullRX order.  A lane takes eight slots with one 16-byte load. */

/* chunks [c0, c1) of wave w of block b, within its list; chunk c of the Border
 * list is chunk P.chI + c in tile numbering */
struct WaveChunks {
    uint32_t c0, c1, slot0, n, tile0;
};
static __device__ __forceinline__ WaveChunks wave_chunks(const GmDev &d, const GmPart &P, uint32_t b, uint32_t w) {
    const bool inB = b >= P.nbI;
    const uint32_t first = ((inB ? b - P.nbI : b) * GM_SW_WAVES + w) * P.cpw, nch = inB ? P.chB : P.chI;
    WaveChunks r;
    r.c0 = first < nch ? first : nch;
    r.c1 = first + P.cpw < nch ? first + P.cpw : nch;
    r.slot0 = inB ? 0u : d.baseI;
    r.n = inB ? d.st->nB : d.st->nI;
    r.tile0 = (inB ? P.chI : 0u) * GM_SW_TPC;
    return r;
}

/* the eight codes of a lane in chunk c, INACTIVE... (0xFFFF) beyond the list's
 * length, and how many of them are occupied */
static __device__ __forceinline__ uint4 chunk_codes(const GmDev &d, const WaveChunks &r, uint32_t c, uint32_t lane,
                                                    uint32_t &nocc) {
    const uint32_t i = c * GM_SW_CHUNK + 8u * lane;
    nocc = r.n > i ? (r.n - i < 8u ? r.n - i : 8u) : 0u;
    return nocc ? *reinterpret_cast<const uint4 *>(d.cstep + r.slot0 + i)
                : make_uint4(0xFFFFFFFFu, 0xFFFFFFFFu, 0xFFFFFFFFu, 0xFFFFFFFFu);
}

static __device__ __forceinline__ uint32_t code_at(const uint4 &cs, int q) {
    const uint32_t wd = q < 2 ? cs.x : q < 4 ? cs.y : q < 6 ? cs.z : cs.w;
    return (wd >> (16 * (q & 1))) & 0xFFFFu;
}

/* the parts into the counts */
__global__ void k_fold_counts(GmDev d) {
    for (uint32_t g = blockIdx.x * blockDim.x + threadIdx.x; g < d.ndefg; g += gridDim.x * blockDim.x) {
        uint32_t v = 0;
#pragma unroll
        for (uint32_t i = 0; i < GM_SUBS; i++) {
            v += d.defsub[(size_t)i * d.ndefg + g];
            d.defsub[(size_t)i * d.ndefg + g] = 0;
        }
        d.defcnt[g] -= v;
    }
}

hipError_t gm_launch_fold_counts(const GmDev &d, hipStream_t s) {
    k_fold_counts<<<fill_blocks(d.ndefg), GM_BLOCK, 0, s>>>(d);
    return hipGetLastError();
}

/* pass 1: per block, the cells that complete in each step of the window and the
 * INACTIVE slots (row GM_WMAX); per wave, the completing cells of each step.
 * Block 0 also clears the window's accumulators.  A slot without a prediction
 * (UNKNOWN) raises GM_ERRF_MISSED. */
__global__ void __launch_bounds__(GM_BLOCK) k_sweep(GmDev d, GmPart P, uint32_t k0, double xcells, uint32_t top_pos) {
    __shared__ uint32_t red[GM_SW_WAVES][GM_WMAX + 1];
    const uint32_t lane = threadIdx.x & 63u, w = threadIdx.x >> 6, b = blockIdx.x;
    if (b == 0 && threadIdx.x == 0) {
        GmStats *st = d.st;
        st->halt = 0;
        st->nexec = 0;
        st->ndeferred = 0;
        st->npend = 0;
        st->pone = 0;
        st->cwrap = 0;
        st->novf = 0;
        st->grow = 0;
        st->need_par = 0;
        st->ticket = 0;
        d.win->nret0 = st->nret;
        d.win->xcells0 = xcells;
        d.win->npend0 = 0;
        d.win->top_hit = 0;
    }
    if (b == 0 && w == 1u && top_pos < d.ndefg) {
        const uint32_t n = exact_count(d, d.rorder[top_pos]);
        if (lane == 0) d.win->left[0] = n;
    }
    const WaveChunks r = wave_chunks(d, P, b, w);
    const uint32_t kc = k0 & (GM_CS_MOD - 1u), horizon = d.horizon;
    uint32_t mine = 0, nrec = 0; /* lane i: step i's cells in the wave */
    bool unknown = false;
    for (uint32_t cb = r.c0; cb < r.c1; cb += GM_SW_PACK) {
        const uint32_t ce = cb + GM_SW_PACK < r.c1 ? cb + GM_SW_PACK : r.c1;
        /* counts of the lane's slots by step, a byte each (at most 8 per chunk) */
        unsigned long long a0 = 0ull, a1 = 0ull;
        for (uint32_t c = cb; c < ce; c++) {
            uint32_t nocc;
            const uint4 cs = chunk_codes(d, r, c, lane, nocc);
#pragma unroll
            for (int q = 0; q < 8; q++) {
                const uint32_t x = code_at(cs, q);
                const bool in = (uint32_t)q < nocc;
                const uint32_t di = (x - kc) & (GM_CS_MOD - 1u);
                const unsigned long long one = in && x < GM_CS_MOD && di < P.W ? 1ull << (8u * (di & 7u)) : 0ull;
                if (di < 8u) a0 += one;
                else a1 += one;
                nrec += in && cs_inactive(x, kc, horizon) ? 1u : 0u;
                unknown |= in && x == GM_CS_UNKNOWN;
            }
        }
        /* wave sums: two 16-bit fields per register (at most 64 * 8 * GM_SW_PACK) */
        uint32_t s[GM_WMAX / 2];
#pragma unroll
        for (int i = 0; i < GM_WMAX / 2; i++) {
            const unsigned long long a = i < 4 ? a0 : a1;
            const uint32_t f = (uint32_t)(a >> (16 * (i & 3))) & 0xFFFFu;
            s[i] = (f & 0xFFu) | (f & 0xFF00u) << 8;
        }
#pragma unroll
        for (int i = 0; i < GM_WMAX / 2; i++) {
            if (2u * i >= P.W) break;
            for (int o = 32; o > 0; o >>= 1) s[i] += (uint32_t)__shfl_xor((int)s[i], o, 64);
            if ((lane >> 1) == (uint32_t)i) mine += (lane & 1u) ? s[i] >> 16 : s[i] & 0xFFFFu;
        }
    }
    for (int o = 32; o > 0; o >>= 1) nrec += __shfl_xor(nrec, o, 64);
    if (__any(unknown) && lane == 0) atomicOr(&d.st->err, GM_ERRF_MISSED);
    if (lane < P.W) {
        red[w][lane] = mine;
        d.wwave[((size_t)b * GM_SW_WAVES + w) * GM_WMAX + lane] = mine;
    }
    if (lane == 0) red[w][GM_WMAX] = nrec;
    __syncthreads();
    const uint32_t t = threadIdx.x;
    if (t < P.W || t == GM_WMAX) {
        uint32_t v = 0;
        for (uint32_t q = 0; q < GM_SW_WAVES; q++) v += red[q][t];
        d.wcnt[(size_t)t * d.swb + b] = v;
    }
}

/* What the window's steps need of the counts' totals: cells completing in step
 * i, where its list starts, the lists' lengths and recyclable slots before step
 * 0.  One thread. */
static __device__ void window_totals(const GmDev &d, const GmPart &P, const uint32_t *tot, uint32_t recI, uint32_t recB,
                                     const uint32_t *totI) {
    GmWin *win = d.win;
    uint32_t off = 0;
    for (uint32_t i = 0; i < P.W; i++) {
        win->full[i] = tot[i];
        win->fullI[i] = totI[i];
        win->off[i] = off;
        off += tot[i];
    }
    win->off[P.W] = off;
    GmWinStep &s = win->step[0];
    s.csz = P.csz0;
    s.nI = d.st->nI;
    s.nB = d.st->nB;
    s.totRecI = recI;
    s.totRecB = recB;
    s.recLenI = recI < d.recCapI ? recI : d.recCapI;
    s.recLenB = recB < d.recCapB ? recB : d.recCapB;
}

/* pass 2, where the window has many blocks (GM_SW_FOLD): one block, a wave
 * per row of counts, 32 consecutive entries per lane; exclusive prefixes over
 * the blocks.  The INACTIVE counts and their prefixes within each list go to the
 * recycling tables of step 0.  (With fewer blocks each block of pass 3 adds up
 * what it needs, which saves this launch: 6 us a step before.) */
__global__ void __launch_bounds__(1024) k_sweep_scan(GmDev d, GmPart P) {
    __shared__ uint32_t stot[GM_WMAX + 1], stotI[GM_WMAX + 1];
    const uint32_t lane = threadIdx.x & 63u, w = threadIdx.x >> 6;
    for (uint32_t row = w; row <= P.W; row += 16u) {
        const bool rec = row == P.W;
        const uint32_t rr = rec ? (uint32_t)GM_WMAX : row;
        const uint32_t *cnt = d.wcnt + (size_t)rr * d.swb;
        uint32_t carry = 0, atI = 0;
        for (uint32_t b0 = 0; b0 < P.nb; b0 += 2048u) {
            const uint32_t i0 = b0 + lane * 32u;
            uint32_t v[32], sum = 0;
#pragma unroll
            for (int i = 0; i < 8; i++) {
                uint4 q = make_uint4(0u, 0u, 0u, 0u);
                if (i0 + 4u * i < P.nb) q = *reinterpret_cast<const uint4 *>(cnt + i0 + 4u * i);
                v[4 * i] = q.x; v[4 * i + 1] = q.y; v[4 * i + 2] = q.z; v[4 * i + 3] = q.w;
            }
#pragma unroll
            for (int i = 0; i < 32; i++) {
                if (i0 + i >= P.nb) v[i] = 0;
                sum += v[i];
            }
            const uint32_t incl = wave_incl_scan(sum);
            uint32_t run = carry + incl - sum;
            /* the prefix at the first Border block */
            const uint32_t atLane = (P.nbI - b0) / 32u;
            uint32_t here = 0;
#pragma unroll
            for (int i = 0; i < 32; i++) {
                const uint32_t x = v[i];
                v[i] = run;
                if (i0 + i == P.nbI) here = run;
                run += x;
            }
            if (P.nbI >= b0 && P.nbI < b0 + 2048u) atI = __shfl(here, (int)atLane, 64);
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const uint32_t b = i0 + 4u * i;
                if (b >= P.nb) continue;
                uint4 q = make_uint4(v[4 * i], v[4 * i + 1], v[4 * i + 2], v[4 * i + 3]);
                if (rec) { /* within the list; the counts themselves are step 0's */
                    *reinterpret_cast<uint4 *>(d.rcnt + b) = *reinterpret_cast<const uint4 *>(cnt + b);
                    *reinterpret_cast<uint4 *>(d.rgone + b) = make_uint4(0u, 0u, 0u, 0u);
                    *reinterpret_cast<uint4 *>(d.rmrg + b) = make_uint4(0u, 0u, 0u, 0u);
                    q.x -= b >= P.nbI ? atI : 0u;
                    q.y -= b + 1u >= P.nbI ? atI : 0u;
                    q.z -= b + 2u >= P.nbI ? atI : 0u;
                    q.w -= b + 3u >= P.nbI ? atI : 0u;
                }
                *reinterpret_cast<uint4 *>((rec ? d.rpre : d.wpre + (size_t)rr * d.swb) + b) = q;
            }
            carry += __shfl(incl, 63, 64);
        }
        if (P.nbI >= P.nb) atI = carry;
        if (lane == 0) {
            stot[row] = carry;
            stotI[row] = atI;
        }
    }
    __syncthreads();
    if (threadIdx.x == 0) window_totals(d, P, stot, stotI[P.W], stot[P.W] - stotI[P.W], stotI);
}

hipError_t gm_launch_reanchor(const GmDev &d, const GmSweepArgs &a, hipStream_t s) {
    k_reanchor<<<grid_for(a.nI + a.nB, GM_BLOCK), GM_BLOCK, 0, s>>>(d, a);
    return hipGetLastError();
}

/* ----------------------------------------------------------------- infection */

/* One pass over the cell grid as it arrived: the cells' (claim, grain) pairs, every word of the bitmap (cells
 * outside the domain stay 0), the cell count of every deformed grain, and whether
 * an id is no deformed grain's (GM_ERRF_GRID).  A thread takes a word, 2 x 16 cells.
 * A wave counts one grain at a time, every lane's cells of it together, and keeps
 * the last grain's sum until another one follows, since atomics on one address are
 * served one after another: a grain met in a long run of words costs few of them
 * (one grain in all: one per block).  The host's two loops over the grid that this
 * replaces took 123 ms at 512^3; the pass takes 0.88, and moves 3.3 GB where the ids,
 * the pairs and the bitmap are 1.6. */
__global__ void __launch_bounds__(GM_BLOCK) k_grid_init(GmDev d, const uint32_t *src, uint32_t nwords) {
    __shared__ uint32_t sid[GM_BLOCK / 64], scnt[GM_BLOCK / 64];
    const uint32_t lane = threadIdx.x & 63u, w = threadIdx.x >> 6;
    const bool vec = (d.nx & 3u) == 0u;
    uint32_t cid = 0xFFFFFFFFu, cn = 0; /* the wave's last grain and its cells not yet added */
    bool bad = false;
    for (uint32_t w0 = blockIdx.x * GM_BLOCK + w * 64u; w0 < nwords; w0 += gridDim.x * GM_BLOCK) {
        const uint32_t wd = w0 + lane;
        const uint32_t line = wd >> 5, sub = wd & 31u;
        const uint32_t bx = line % d.dnbx, rest = line / d.dnbx, by = rest % d.dnby, bz = rest / d.dnby;
        const uint32_t x0 = bx * 16u, y0 = by * 8u + 2u * (sub & 3u), z = bz * 8u + (sub >> 2);
        uint32_t id[32], in = 0, v = 0;
#pragma unroll
        for (uint32_t r = 0; r < 2u; r++) {
            const bool row = wd < nwords && y0 + r < d.ny && z < d.nz;
            const size_t at = x0 + (size_t)(y0 + r) * d.nx + (size_t)z * d.nxy;
            const uint32_t *g = src + at;
            uint2 *c = d.cell + at;
#pragma unroll
            for (uint32_t i = 0; i < 16u; i += 4u) {
                uint4 q = make_uint4(0u, 0u, 0u, 0u);
                if (vec) {
                    if (row && x0 + i < d.nx) q = *reinterpret_cast<const uint4 *>(g + i);
                } else if (row) {
                    if (x0 + i < d.nx) q.x = g[i];
                    if (x0 + i + 1u < d.nx) q.y = g[i + 1u];
                    if (x0 + i + 2u < d.nx) q.z = g[i + 2u];
                    if (x0 + i + 3u < d.nx) q.w = g[i + 3u];
                }
                if (vec) {
                    if (row && x0 + i < d.nx) {
                        uint4 *o = reinterpret_cast<uint4 *>(c + i);
                        o[0] = make_uint4(GM_FREE_CLAIM, q.x, GM_FREE_CLAIM, q.y);
                        o[1] = make_uint4(GM_FREE_CLAIM, q.z, GM_FREE_CLAIM, q.w);
                    }
                } else if (row) {
                    if (x0 + i < d.nx) c[i] = make_uint2(GM_FREE_CLAIM, q.x);
                    if (x0 + i + 1u < d.nx) c[i + 1u] = make_uint2(GM_FREE_CLAIM, q.y);
                    if (x0 + i + 2u < d.nx) c[i + 2u] = make_uint2(GM_FREE_CLAIM, q.z);
                    if (x0 + i + 3u < d.nx) c[i + 3u] = make_uint2(GM_FREE_CLAIM, q.w);
                }
                const uint32_t k = 16u * r + i;
                id[k] = q.x;
                id[k + 1] = q.y;
                id[k + 2] = q.z;
                id[k + 3] = q.w;
#pragma unroll
                for (uint32_t e = 0; e < 4u; e++) in |= row && x0 + i + e < d.nx ? 1u << (k + e) : 0u;
            }
        }
#pragma unroll
        for (int i = 0; i < 32; i++) v |= id[i] < d.ndefg ? 1u << i : 0u;
        v &= in;
        bad |= v != in;
        if (wd < nwords) d.dmap[wd] = v;
        /* distinct grains of the wave's words */
        for (uint32_t left = v;;) {
            const uint64_t any = __ballot(left != 0u);
            if (!any) break;
            uint32_t cand = 0;
#pragma unroll
            for (int i = 31; i >= 0; i--) cand = (left >> i) & 1u ? id[i] : cand;
            const uint32_t g = rdlane(cand, (uint32_t)__ffsll((long long)any) - 1u);
            uint32_t hit = 0;
#pragma unroll
            for (int i = 0; i < 32; i++) hit |= id[i] == g ? 1u << i : 0u;
            hit &= left;
            left &= ~hit;
            uint32_t n = (uint32_t)__popc(hit);
            for (int o = 32; o > 0; o >>= 1) n += (uint32_t)__shfl_xor((int)n, o, 64);
            if (g != cid) {
                if (lane == 0 && cn) atomicAdd(&d.defcnt[cid], cn);
                cid = g;
                cn = 0;
            }
            cn += n;
        }
    }
    if (__any(bad) && lane == 0) atomicOr(&d.st->err, GM_ERRF_GRID);
    /* the waves' last grains, equal ones together */
    if (lane == 0) {
        sid[w] = cid;
        scnt[w] = cn;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (uint32_t i = 0; i < GM_BLOCK / 64u; i++) {
            uint32_t n = scnt[i];
            if (!n) continue;
            for (uint32_t q = i + 1u; q < GM_BLOCK / 64u; q++)
                if (scnt[q] && sid[q] == sid[i]) {
                    n += scnt[q];
                    scnt[q] = 0;
                }
            atomicAdd(&d.defcnt[sid[i]], n);
        }
    }
}

hipError_t gm_launch_grid_init(const GmDev &d, const uint32_t *src, hipStream_t s) {
    const uint32_t nwords = d.dnbx * d.dnby * d.dnbz * 32u;
    const unsigned nb = fill_blocks(nwords);
    k_grid_init<<<nb < GM_GRID_BLOCKS ? nb : GM_GRID_BLOCKS, GM_BLOCK, 0, s>>>(d, src, nwords);
    return hipGetLastError();
}

/* Target of attempt rank r from a parent at (x,y,z).  Inside parents
 * (omp_infect_OutOfRXFrontInside, SCORE_Kernel.cpp:4252-4344) never wrap; they send
 * every target to the Border list unless they lie more than one cell away from
 * every face (:4606-4609).  Border parents (:4347-4493) wrap x and y, drop
 * targets outside z, and send strictly interior targets to the Inside list. */
static __device__ __forceinline__ bool attempt_target(const GmDev &d, bool fromB, uint32_t x, uint32_t y, uint32_t z,
                                                      int r, uint32_t &tx_, uint32_t &ty_, uint32_t &tz_, bool &toB) {
    int tx = (int)x + dir_dx(r), ty = (int)y + dir_dy(r), tz = (int)z + dir_dz(r);
    const int nx = (int)d.nx, ny = (int)d.ny, nz = (int)d.nz;
    if (fromB) {
        if (tx < 0) tx += nx;
        if (tx >= nx) tx -= nx;
        if (ty < 0) ty += ny;
        if (ty >= ny) ty -= ny;
        if (tz < 0 || tz >= nz) return false;
        toB = !(tx > 0 && tx < nx - 1 && ty > 0 && ty < ny - 1 && tz > 0 && tz < nz - 1);
    } else {
        /* Inside cells are strictly interior, so this never fires; it keeps a
         * corrupted record from addressing outside the grid */
        if (tx < 0 || tx >= nx || ty < 0 || ty >= ny || tz < 0 || tz >= nz) return false;
        toB = !((int)x > 1 && (int)x < nx - 2 && (int)y > 1 && (int)y < ny - 2 && (int)z > 1 && (int)z < nz - 2);
    }
    tx_ = (uint32_t)tx;
    ty_ = (uint32_t)ty;
    tz_ = (uint32_t)tz;
    return true;
}


/* sum over the block (GM_BLOCK threads) of three values; every thread gets them */
static __device__ __forceinline__ void block_sum3(uint32_t &a, uint32_t &b, uint32_t &c, uint32_t (*sh)[3]) {
    for (int o = 32; o > 0; o >>= 1) {
        a += __shfl_xor(a, o, 64);
        b += __shfl_xor(b, o, 64);
        c += __shfl_xor(c, o, 64);
    }
    const uint32_t w = threadIdx.x >> 6;
    __syncthreads();
    if ((threadIdx.x & 63u) == 0) {
        sh[w][0] = a;
        sh[w][1] = b;
        sh[w][2] = c;
    }
    __syncthreads();
    a = b = c = 0;
#pragma unroll
    for (int i = 0; i < GM_BLOCK / 64; i++) {
        a += sh[i][0];
        b += sh[i][1];
        c += sh[i][2];
    }
}

/* blocks that counted step j's attempts */
static __device__ __forceinline__ uint32_t attempt_blocks(const GmPart &P, uint32_t j) {
    return j == 0u && P.fused ? P.nb : P.nbp;
}

/* Closes step js of the window, by one block after the step's commit pass: its
 * row for the host's master section, the lists' lengths and, with `next`, the
 * recycling tables of step js+1: per sweep block, how many of its INACTIVE slots
 * step js handed out (the first min(winners, cap) of each list, ascending), how
 * many it has now that step js's completed cells are INACTIVE, and their prefix
 * within the list. */
static __device__ void close_step(const GmDev &d, const GmPart &P, uint32_t js, bool next) {
    __shared__ uint32_t sh[GM_BLOCK / 64][3];
    __shared__ unsigned long long ws[GM_BLOCK / 64];
    GmStats *st = d.st;
    GmWin *win = d.win;
    const uint32_t t = threadIdx.x, lane = t & 63u, w = t >> 6;
    const uint32_t rp = (js & 1u) * d.swb, rn = ((js + 1u) & 1u) * d.swb;
    /* every load that needs no other's result is issued before the first is waited for:
     * with six round trips in a row this block, not the parents', was the propose
     * pass's longest */
    static_assert(GM_DB <= 4 * GM_BLOCK && GM_PB <= 8 * GM_BLOCK, "one round of loads each");
    uint2 bt[4];
#pragma unroll
    for (uint32_t i = 0; i < 4u; i++) bt[i] = t + i * GM_BLOCK < P.nbd ? d.btot[t + i * GM_BLOCK] : make_uint2(0u, 0u);
    uint32_t ac[8];
    const uint32_t *acnt = d.acnt + (js & 1u) * GM_PB, nba = attempt_blocks(P, js);
#pragma unroll
    for (uint32_t i = 0; i < 8u; i++) ac[i] = t + i * GM_BLOCK < nba ? acnt[t + i * GM_BLOCK] : 0u;
    uint32_t R[8], pre[8], full[8];
    auto tables = [&](uint32_t i0) {
        if (i0 >= P.nb) return;
        const uint4 *q = reinterpret_cast<const uint4 *>(d.rcnt + rp + i0);
        const uint4 *u = reinterpret_cast<const uint4 *>(d.rpre + rp + i0);
        const uint4 *f = reinterpret_cast<const uint4 *>(d.wcnt + (size_t)js * d.swb + i0);
        const uint4 q0 = q[0], q1 = q[1], u0 = u[0], u1 = u[1], f0 = f[0], f1 = f[1];
        R[0] = q0.x; R[1] = q0.y; R[2] = q0.z; R[3] = q0.w; R[4] = q1.x; R[5] = q1.y; R[6] = q1.z; R[7] = q1.w;
        pre[0] = u0.x; pre[1] = u0.y; pre[2] = u0.z; pre[3] = u0.w;
        pre[4] = u1.x; pre[5] = u1.y; pre[6] = u1.z; pre[7] = u1.w;
        full[0] = f0.x; full[1] = f0.y; full[2] = f0.z; full[3] = f0.w;
        full[4] = f1.x; full[5] = f1.y; full[6] = f1.z; full[7] = f1.w;
    };
    if (next) tables(8u * t);
    const GmWinStep o = win->step[js];
    GmStepRow r;
    r.nfullI = win->fullI[js];
    const uint32_t nfull = win->full[js], npend = agent_load(&st->npend), npend0 = win->npend0;
    r.err = agent_load(&st->err);
    r.pone = agent_load(&st->pone);
    r.nplaced = st->nplaced;
    r.pkey = st->arr_pkey;
    const unsigned long long nret = st->nret;
    uint32_t wI = bt[0].x + bt[1].x + bt[2].x + bt[3].x, wB = bt[0].y + bt[1].y + bt[2].y + bt[3].y;
    uint32_t na = ac[0] + ac[1] + ac[2] + ac[3] + ac[4] + ac[5] + ac[6] + ac[7];
    block_sum3(wI, wB, na, sh);
    const uint32_t limI = wI < o.recLenI ? wI : o.recLenI, limB = wB < o.recLenB ? wB : o.recLenB;
    unsigned long long carry = 0ull; /* Inside | Border totals */
    if (next) {
        for (uint32_t b0 = 0; b0 < P.nb; b0 += 8u * GM_BLOCK) {
            const uint32_t i0 = b0 + 8u * t;
            if (b0) tables(i0);
            unsigned long long sum = 0ull;
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const uint32_t b = i0 + i;
                if (b >= P.nb) {
                    R[i] = pre[i] = 0;
                    continue;
                }
                const uint32_t lim = b < P.nbI ? limI : limB;
                const uint32_t left = pre[i] < lim ? lim - pre[i] : 0u;
                pre[i] = left < R[i] ? left : R[i]; /* handed out */
                R[i] = R[i] - pre[i] + full[i];
                sum += b < P.nbI ? (unsigned long long)R[i] << 32 : (unsigned long long)R[i];
            }
            unsigned long long incl = sum;
            for (int s = 1; s < 64; s <<= 1) {
                const unsigned long long v = (unsigned long long)__shfl_up((long long)incl, s, 64);
                if (lane >= (uint32_t)s) incl += v;
            }
            __syncthreads();
            if (lane == 63u) ws[w] = incl;
            __syncthreads();
            unsigned long long before = carry + incl - sum;
            for (uint32_t i = 0; i < GM_BLOCK / 64; i++) {
                if (i < w) before += ws[i];
                carry += ws[i];
            }
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const uint32_t b = i0 + i;
                if (b >= P.nb) break;
                d.rgone[b] = pre[i];
                d.rcnt[rn + b] = R[i];
                d.rpre[rn + b] = b < P.nbI ? (uint32_t)(before >> 32) : (uint32_t)before;
                before += b < P.nbI ? (unsigned long long)R[i] << 32 : (unsigned long long)R[i];
            }
        }
    }
    if (t != 0) return;
    r.nI = o.nI + (wI - limI);
    r.nB = o.nB + (wB - limB);
    r.nfullB = nfull - r.nfullI;
    r.totRecI = o.totRecI;
    r.totRecB = o.totRecB;
    r.recLenI = o.recLenI;
    r.recLenB = o.recLenB;
    r.winI = wI;
    r.winB = wB;
    r.npend = npend - npend0;
    r.nattempt = na;
    st->rows[js] = r;
    st->nplaced = 0;
    st->pone = 0;
    st->arr_pkey = 0ull;
    win->npend0 = npend;
    st->nI = r.nI;
    st->nB = r.nB;
    st->nret = nret + (unsigned long long)nfull;
    st->nexec = js + 1u;
    if (next) {
        GmWinStep &s = win->step[js + 1u];
        s.csz = gm_chunk_size(nfull, wI + wB);
        s.nI = r.nI;
        s.nB = r.nB;
        s.totRecI = (uint32_t)(carry >> 32);
        s.totRecB = (uint32_t)carry;
        s.recLenI = s.totRecI < d.recCapI ? s.totRecI : d.recCapI;
        s.recLenB = s.totRecB < d.recCapB ? s.totRecB : d.recCapB;
    }
}

/* Why step j of the window must not run.  HOST: the host has to act on what step j-1
 * left (an error, a count that wrapped, the exhaustion of the grain that sets rhomax,
 * Xcells at a threshold, weights the window cannot wait for, a step that found too few
 * slots).  Else an error of the step's own: infection keys are p*32 + rank in 32 bits, p
 * below its nfull parents, and the retirement log, of which it takes the entries from
 * `ret` on, has an end.  Else PLANES: it has more parents than the planes hold.
 * The inputs were written by earlier kernels, but for st->err, to which block 0 of the
 * propose pass adds only where every block finds one of the step's own errors: all
 * blocks halt, or none.  Block 0 records it in st->halt for the step's other passes and
 * for the steps queued behind it, which do nothing then. */
#define HALT_HOST 0x80000000u
#define HALT_PLANES 0x40000000u
#define HALT_ERRF (GM_ERRF_KEYS | GM_ERRF_RLOG_FULL)
static __device__ __forceinline__ uint32_t halt_reason(const GmDev &d, const GmWindow &w, uint32_t nfull,
                                                       unsigned long long ret, bool at_stop) {
    const GmStats *st = d.st;
    /* every word loaded before the first test */
    const uint32_t flags = either_load(&st->err) | st->cwrap | st->novf | d.win->top_hit | st->grow, npend = st->npend;
    const bool host = (flags != 0u) | ((npend != 0u) & !w.defer) | (npend > w.pend_limit) | at_stop;
    const uint32_t err = (nfull > (1u << 27) ? GM_ERRF_KEYS : 0u) | (ret + nfull > d.rlogCap ? GM_ERRF_RLOG_FULL : 0u);
    return host ? HALT_HOST : err ? err : nfull > d.parentCap ? HALT_PLANES : 0u;
}
/* by one thread of block 0 */
static __device__ __forceinline__ void record_halt(const GmDev &d, uint32_t why, uint32_t nfull, uint32_t j) {
    d.st->halt = why ? 1u : 0u;
    if (why & HALT_PLANES) d.st->need_par = nfull;
    if (why & HALT_ERRF) atomicOr(&d.st->err, why);
    if (d.prog) __hip_atomic_store(d.prog, (j << 1) | (why ? 1u : 0u), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

/* Step k's parent p, in slot s: see k_propose; returns its attempts.  rlog: where the
 * step's retirements go in the log. */
static __device__ __forceinline__ uint32_t propose_parent(const GmDev &d, uint32_t s, uint32_t p, uint32_t k, uint2 *rlog) {
    const GmRec *r = d.rec + s;
    const RecC rc = rec_c(r);
    const RecA ra = rec_a(r);
    const double inc = r->inc;
    const uint32_t rxg = r->rxg, cell = rc.cell;
    const uint32_t z = cell / d.nxy, rem = cell - z * d.nxy, y = rem / d.nx, x = rem - y * d.nx;
    const bool fromB = s < d.baseI;
    const bool interior = (x - 1u < d.nx - 2u) & (y - 1u < d.ny - 2u) & (z - 1u < d.nz - 2u);
    Neighbourhood nb;
    if (interior) nb.load(d, x, y, z);
    /* rxFrac after the completing addition, while the bits are on their way */
    const double fin = advanced(ra.frac0, inc, k - ra.s0 + 1u);
    const uint32_t am = interior ? nb.mask() : face_attempts(d, x, y, z);
    for (uint32_t m = am; m; m &= m - 1u) {
        const uint32_t rk = (uint32_t)__ffs(m) - 1u;
        uint32_t t = cell + (uint32_t)(dir_dx(rk) + dir_dy(rk) * (int)d.nx + dir_dz(rk) * (int)d.nxy);
        if (!interior) {
            uint32_t tx, ty, tz;
            bool toB;
            attempt_target(d, true, x, y, z, (int)rk, tx, ty, tz, toB);
            t = cell_of(d, tx, ty, tz);
        }
        atomicMin(&d.cell[t].x, p * 32u + rk);
    }
    d.pmA[p] = am;
    par_plane(d, GM_PAR1_CELL)[p] = make_uint4(x | y << 16, z | (fromB ? 1u << 16 : 0u), rc.defg, rxg);
    reinterpret_cast<double2 *>(par_plane(d, GM_PAR1_FP))[p] = make_double2(fin, rc.P);
    rlog[p] = make_uint2(cell, d.ndefg + rxg);
    return (uint32_t)__popc(am);
}

/* Step j's attempts, one lane per parent.  What the infection needs of the parent
 * goes to the dense parent planes (FullRX order), with its rxFrac after the
 * completing addition, replayed from the anchor.  Every attempt on a deformed cell
 * claims its target (the smallest key p*32+r is the serial winner); their mask
 * over the ranks is kept in pmA for the decide pass.  Few of the 26 neighbours are
 * still deformed (1.04 per parent on the 512^3 workload), so the cost is finding
 * them: a strictly interior parent reads its 3x3x3 bits with three 16-byte loads
 * (26 single tests before).  Wave w
 * of a block takes chunks of 64 parents w*nbp apart, so that a short list spreads
 * over the CUs.  Block 0 closes the step before. */
__global__ void __launch_bounds__(GM_BLOCK) k_propose(GmDev d, GmPart P, GmWindow wd, uint32_t j, uint32_t k) {
    __shared__ uint32_t satt[GM_BLOCK / 64];
    GmStats *st = d.st;
    const GmWin *win = d.win;
    const uint32_t nfull = win->full[j], off = win->off[j];
    /* the window may have halted at an earlier step: the one before this did not run, and
     * nothing is left to close.  (Block 0 sets the word only where every block halts.) */
    const uint32_t halted = either_load(&st->halt);
    const unsigned long long nret = win->nret0 + off;
    const uint32_t halt = halt_reason(d, wd, nfull, nret, (j != 0u) & (win->xcells0 + (double)off >= wd.xstop));
    if (halted) return;
    if (blockIdx.x == 0) {
        /* a step whose commit pass found too few slots is not done */
        const uint32_t undone = st->grow;
        if (j && !undone) close_step(d, P, j - 1u, !halt);
        if (threadIdx.x == 0) record_halt(d, halt, nfull, j);
        return;
    }
    if (halt) return;
    /* the step's parents retire into the log at [nret, nret + nfull) */
    uint2 *rlog = d.rlog + nret;
    const uint32_t blk = blockIdx.x - 1u, lane = threadIdx.x & 63u, w = threadIdx.x >> 6;
    uint32_t natt = 0;
    for (uint32_t c = w * P.nbp + blk; c * 64u < nfull; c += P.nbp * (GM_BLOCK / 64u)) {
        const uint32_t p = c * 64u + lane;
        if (p >= nfull) break;
        natt += propose_parent(d, d.pslot[off + p], p, k, rlog);
    }
    for (int o = 32; o > 0; o >>= 1) natt += __shfl_xor(natt, o, 64);
    if (lane == 0) satt[w] = natt;
    __syncthreads();
    if (threadIdx.x == 0) d.acnt[(j & 1u) * GM_PB + blk] = satt[0] + satt[1] + satt[2] + satt[3];
}

/* pass 3: append_to_fullrx_*_list (SCORE_Kernel.cpp:3994-4042, :4133-4180) of
 * every step as ordered compaction: step i's completed slots ascending, Inside
 * then Border, at pslot[win->off[i]...]; and the INACTIVE mask of every 64-slot
 * tile, from which the steps hand out recycled slots.  FOLD: the block adds up
 * the counts of the blocks itself.  PROPOSE: the blocks then take the first step's
 * parents they have listed through the propose pass, which saves a launch a window: 5 us
 * of every step where the scalars change in each. */
template <bool FOLD, bool PROPOSE>
__global__ void __launch_bounds__(GM_BLOCK) k_compact(GmDev d, GmPart P, GmWindow wd, uint32_t k0) {
    __shared__ uint32_t stot[GM_WMAX + 1], spre[GM_WMAX + 1], stotI[GM_WMAX + 1], base[GM_WMAX];
    __shared__ uint32_t run[GM_SW_WAVES][GM_WMAX];
    __shared__ uint64_t sR[GM_SW_WAVES][8];
    /* per lane 16 counters of 16 bits, rows of 40 bytes against bank conflicts */
    __shared__ __align__(8) uint32_t sl[GM_SW_WAVES][64][10];
    const uint32_t lane = threadIdx.x & 63u, w = threadIdx.x >> 6, b = blockIdx.x, t = threadIdx.x;
    if (FOLD) {
        for (uint32_t row = w; row <= P.W; row += GM_SW_WAVES) {
            const bool rec = row == P.W;
            const uint32_t *cnt = d.wcnt + (size_t)(rec ? (uint32_t)GM_WMAX : row) * d.swb;
            uint32_t a = 0, p = 0, pI = 0;
            for (uint32_t i0 = 4u * lane; i0 < P.nb; i0 += 256u) {
                const uint4 q = *reinterpret_cast<const uint4 *>(cnt + i0);
                const uint32_t v[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
                for (uint32_t i = 0; i < 4; i++) {
                    const uint32_t x = i0 + i < P.nb ? v[i] : 0u;
                    a += x;
                    p += i0 + i < b ? x : 0u;
                    pI += i0 + i < P.nbI ? x : 0u;
                }
            }
            for (int o = 32; o > 0; o >>= 1) {
                a += __shfl_xor(a, o, 64);
                p += __shfl_xor(p, o, 64);
                pI += __shfl_xor(pI, o, 64);
            }
            if (lane == 0) {
                stot[row] = a;
                spre[row] = p;
                stotI[row] = pI;
            }
        }
        __syncthreads();
        if (t < P.W) {
            uint32_t o = spre[t];
            d.wpre[(size_t)t * d.swb + b] = o;
            for (uint32_t i = 0; i < t; i++) o += stot[i];
            base[t] = o;
        }
        if (t == GM_WMAX) {
            d.rcnt[b] = d.wcnt[(size_t)GM_WMAX * d.swb + b];
            d.rpre[b] = spre[P.W] - (b >= P.nbI ? stotI[P.W] : 0u);
            d.rgone[b] = 0;
            d.rmrg[b] = 0;
        }
        if (b == 0 && t == 64u) window_totals(d, P, stot, stotI[P.W], stot[P.W] - stotI[P.W], stotI);
    } else if (t < P.W) {
        base[t] = d.win->off[t] + d.wpre[(size_t)t * d.swb + b];
    }
    __syncthreads();
    if (lane < P.W) {
        uint32_t o = base[lane];
        const uint32_t *ww = d.wwave + (size_t)b * GM_SW_WAVES * GM_WMAX + lane;
        for (uint32_t q = 0; q < w; q++) o += ww[q * GM_WMAX];
        run[w][lane] = o;
    }
    wave_sync();
    const WaveChunks r = wave_chunks(d, P, b, w);
    const uint32_t kc = k0 & (GM_CS_MOD - 1u), horizon = d.horizon;
    for (uint32_t c = r.c0; c < r.c1; c++) {
        uint32_t nocc;
        const uint4 cs = chunk_codes(d, r, c, lane, nocc);
        unsigned long long cnt = 0ull; /* 16 counters of 4 bits (at most 8 each) */
        uint32_t full = 0, rec = 0;
#pragma unroll
        for (int q = 0; q < 8; q++) {
            const uint32_t x = code_at(cs, q);
            const bool in = (uint32_t)q < nocc;
            const uint32_t di = (x - kc) & (GM_CS_MOD - 1u);
            const bool f = in && x < GM_CS_MOD && di < P.W;
            cnt += f ? 1ull << (4u * (di & 15u)) : 0ull;
            full |= f ? 1u << q : 0u;
            rec |= in && cs_inactive(x, kc, horizon) ? 1u << q : 0u;
        }
        reinterpret_cast<uint8_t *>(sR[w])[lane] = (uint8_t)rec;
        wave_sync();
        if (lane < GM_SW_TPC) d.mR[r.tile0 + c * GM_SW_TPC + lane] = sR[w][lane];
        if (!__any(full != 0u)) {
            wave_sync();
            continue;
        }
        uint32_t incl[GM_WMAX / 2];
#pragma unroll
        for (int i = 0; i < GM_WMAX / 2; i++) {
            if (2u * i >= P.W) break;
            const uint32_t f = (uint32_t)(cnt >> (8 * i));
            const uint32_t v = (f & 0xFu) | (f & 0xF0u) << 12;
            incl[i] = wave_incl_scan(v);
            sl[w][lane][i] = incl[i] - v;
        }
        wave_sync();
        uint16_t *mineRow = reinterpret_cast<uint16_t *>(sl[w][lane]);
        const uint32_t slot = r.slot0 + c * GM_SW_CHUNK + 8u * lane;
#pragma unroll
        for (int q = 0; q < 8; q++) {
            if (!((full >> q) & 1u)) continue;
            const uint32_t di = (code_at(cs, q) - kc) & (GM_CS_MOD - 1u);
            const uint32_t o = mineRow[di];
            mineRow[di] = (uint16_t)(o + 1u);
            d.pslot[run[w][di] + o] = slot + (uint32_t)q;
        }
        wave_sync();
        if (lane == 63u) {
#pragma unroll
            for (int i = 0; i < GM_WMAX / 2; i++) {
                if (2u * i >= P.W) break;
                run[w][2 * i] += incl[i] & 0xFFFFu;
                run[w][2 * i + 1] += incl[i] >> 16;
            }
        }
        wave_sync();
    }
    if (!PROPOSE) return;
    /* the first step's attempts by the blocks that list its parents */
    const uint32_t nfull = stot[0], first = spre[0], cnt = d.wcnt[b];
    const unsigned long long nret = d.st->nret;
    const uint32_t halt = halt_reason(d, wd, nfull, nret, false);
    if (b == 0 && t == 0) record_halt(d, halt, nfull, 0u);
    if (halt) return;
    __syncthreads();
    uint32_t natt = 0;
    for (uint32_t i = t; i < cnt; i += GM_BLOCK)
        natt += propose_parent(d, d.pslot[first + i], first + i, k0, d.rlog + nret);
    for (int o = 32; o > 0; o >>= 1) natt += __shfl_xor(natt, o, 64);
    if (lane == 0) run[w][0] = natt;
    __syncthreads();
    if (t == 0) d.acnt[b] = run[0][0] + run[1][0] + run[2][0] + run[3][0];
}

__global__ void k_arrivals(GmDev d, GmSweepArgs A);

hipError_t gm_launch_window(const GmDev &d, const GmPart &P, const GmSweepArgs &a, const GmWindow &wd, bool arrivals,
                            double xcells, hipStream_t s, hipEvent_t *ev) {
    hipError_t e;
    if ((e = mark(ev, 0, s)) != hipSuccess) return e;
    if (a.reanchor && (e = gm_launch_reanchor(d, a, s)) != hipSuccess) return e;
    if (arrivals) {
        k_arrivals<<<1, 1024, 0, s>>>(d, a);
        if ((e = hipGetLastError()) != hipSuccess) return e;
    }
    if ((e = mark(ev, 1, s)) != hipSuccess) return e;
    k_sweep<<<P.nb, GM_BLOCK, 0, s>>>(d, P, a.k, xcells, wd.top_pos);
    if ((e = mark(ev, 2, s)) != hipSuccess) return e;
    const bool fold = gm_fold(P);
    if (!fold) k_sweep_scan<<<1, 1024, 0, s>>>(d, P);
    if ((e = mark(ev, 3, s)) != hipSuccess) return e;
    if (P.fused) k_compact<true, true><<<P.nb, GM_BLOCK, 0, s>>>(d, P, wd, a.k);
    else if (fold) k_compact<true, false><<<P.nb, GM_BLOCK, 0, s>>>(d, P, wd, a.k);
    else k_compact<false, false><<<P.nb, GM_BLOCK, 0, s>>>(d, P, wd, a.k);
    return hipGetLastError();
}

/* exclusive prefix of v over the block (GM_BLOCK threads) and the total */
static __device__ __forceinline__ uint32_t block_excl_scan(uint32_t v, uint32_t *sh, uint32_t &tot) {
    const uint32_t incl = wave_incl_scan(v), w = threadIdx.x >> 6;
    __syncthreads();
    if ((threadIdx.x & 63u) == 63u) sh[w] = incl;
    __syncthreads();
    uint32_t pre = 0;
    tot = 0;
#pragma unroll
    for (uint32_t i = 0; i < GM_BLOCK / 64; i++) {
        if (i < w) pre += sh[i];
        tot += sh[i];
    }
    return pre + incl - v;
}

/* append_to_recycling_*_list (SCORE_Kernel.cpp:4037-4041, :4175-4179): the
 * recycled slots in ascending order, of which only the first min(winners, cap)
 * are ever handed out.  Runs beside the decide pass, so the winners are not
 * counted yet: their upper bound is the step's attempts (1.03 per winner).  A
 * block takes sweep blocks r, r + nrec, ... and keeps their INACTIVE masks up to
 * date within the window: the slots the step before handed out leave (the first
 * rgone of them), the cells completed since the masks were last brought up to date
 * join, and the part of the slots that lies below the bound is written.  Sweep
 * blocks beyond it are left alone and catch up when they are reached. */
static __device__ void recycle_blocks(const GmDev &d, const GmPart &P, uint32_t j, uint32_t r, uint32_t nrec,
                                      unsigned long long *sm) {
    __shared__ uint32_t sh[GM_BLOCK / 64], sn[GM_BLOCK / 64][3], sfull[GM_WMAX], slist[GM_WMAX];
    const GmWin *win = d.win;
    const uint32_t t = threadIdx.x, lane = t & 63u, w = t >> 6;
    const uint32_t rp = (j & 1u) * d.swb, nt = GM_SW_WAVES * P.cpw * GM_SW_TPC;
    uint32_t *so = reinterpret_cast<uint32_t *>(sm + nt);
    const uint32_t recI = win->step[j].recLenI, recB = win->step[j].recLenB;
    const uint32_t halt = d.st->halt, nba = attempt_blocks(P, j);
    uint32_t na = 0, z0 = 0, z1 = 0;
    uint4 ac[2];
    static_assert(GM_PB <= 8 * GM_BLOCK, "one round of loads");
#pragma unroll
    for (uint32_t i = 0; i < 2u; i++) {
        ac[i] = make_uint4(0u, 0u, 0u, 0u);
        const uint32_t at = 4u * (t + i * GM_BLOCK);
        if (at < nba) ac[i] = *reinterpret_cast<const uint4 *>(d.acnt + (j & 1u) * GM_PB + at);
    }
    for (uint32_t b = r; b < P.nb; b += nrec) {
        /* everything a block may need is loaded before its first use: its masks, what the
         * step before handed out, where each step's completed cells are listed */
        const bool inB = b >= P.nbI;
        const uint32_t nch = inB ? P.chB : P.chI, ch0 = (inB ? b - P.nbI : b) * GM_SW_WAVES * P.cpw;
        const uint32_t n = (ch0 + GM_SW_WAVES * P.cpw < nch ? GM_SW_WAVES * P.cpw : nch - ch0) * GM_SW_TPC;
        const uint32_t t0 = ((inB ? P.chI : 0u) + ch0) * GM_SW_TPC;
        const unsigned long long m0 = t < n ? d.mR[t0 + t] : 0ull;
        const uint32_t merged = d.rmrg[b], pre = d.rpre[rp + b], gone = j ? d.rgone[b] : 0u, rec = inB ? recB : recI;
        uint32_t lf = 0, lo = 0;
        if (t < j) {
            lf = d.wcnt[(size_t)t * d.swb + b];
            lo = win->off[t] + d.wpre[(size_t)t * d.swb + b];
        }
        if (b == r) {
#pragma unroll
            for (uint32_t i = 0; i < 2u; i++) {
                const uint32_t at = 4u * (t + i * GM_BLOCK);
                na += ac[i].x + (at + 1u < nba ? ac[i].y : 0u) + (at + 2u < nba ? ac[i].z : 0u) + (at + 3u < nba ? ac[i].w : 0u);
            }
            block_sum3(na, z0, z1, sn);
            if (halt) return;
        }
        const uint32_t bound = na < rec ? na : rec;
        if (gone == 0u && pre >= bound) continue;
        const uint32_t rel0 = ch0 * GM_SW_CHUNK, slot0 = (inB ? 0u : d.baseI) + rel0;
        uint32_t run = 0;
        __syncthreads();
        if (t < j) {
            sfull[t] = lf;
            slist[t] = lo;
        }
        for (uint32_t i0 = 0; i0 < n; i0 += GM_BLOCK) {
            const uint32_t i = i0 + t;
            unsigned long long m = i0 == 0u ? m0 : i < n ? d.mR[t0 + i] : 0ull;
            if (run < gone) {
                const uint32_t c = (uint32_t)__popcll(m);
                uint32_t tot;
                const uint32_t before = run + block_excl_scan(c, sh, tot);
                if (before + c <= gone) m = 0ull;
                else
                    for (uint32_t q = before < gone ? gone - before : 0u; q; q--) m &= m - 1ull;
                run += tot;
            }
            if (i < n) sm[i] = m;
        }
        __syncthreads();
        for (uint32_t i = merged; i < j; i++) {
            const uint32_t nf = sfull[i];
            const uint32_t *list = d.pslot + slist[i];
            for (uint32_t q = t; q < nf; q += GM_BLOCK) {
                const uint32_t s = list[q] - slot0;
                atomicOr(&sm[s >> 6], 1ull << (s & 63u));
            }
        }
        __syncthreads();
        run = pre;
        for (uint32_t i0 = 0; i0 < n; i0 += GM_BLOCK) {
            const uint32_t i = i0 + t;
            const unsigned long long m = i < n ? sm[i] : 0ull;
            if (i < n) d.mR[t0 + i] = m;
            uint32_t tot;
            const uint32_t o = run + block_excl_scan((uint32_t)__popcll(m), sh, tot);
            if (i < n) so[i] = o;
            run += tot;
        }
        if (t == 0) d.rmrg[b] = j;
        __syncthreads();
        /* tile by tile, a lane per slot */
        uint32_t *out = inB ? d.recB : d.recI;
        for (uint32_t i = w; i < n; i += GM_SW_WAVES) {
            const unsigned long long m = sm[i];
            const uint32_t o = so[i];
            if (o >= bound) break;
            const uint32_t q = o + lanemask_lt_count(m);
            if ((m >> lane & 1ull) && q < bound) out[q] = rel0 + 64u * i + lane;
        }
    }
}

/* The first nrec blocks write the recycled slots; the rest find which attempts
 * won.  A wave takes a chunk of parents at a time and flattens their attempts into
 * a list, a lane per attempt, so that all claims are loaded together (a loop over
 * each parent's attempts waits once per attempt of its busiest parent).  A cell's
 * claim and grain are one 8-byte load; the grains go to the commit pass in the
 * attempts' order (the first GM_GATT of a chunk), which would wait for the same
 * scattered lines again.  Winners as 26-bit masks per destination list, their
 * counts per chunk (Inside << 16 | Border) and per block, from which the commit
 * pass ranks them.  The parents retire here (updateFullRX*, SCORE_Kernel.cpp:
 * 4640-4653), beside the waiting for the claims. */
__global__ void __launch_bounds__(GM_BLOCK) k_decide(GmDev d, GmPart P, uint32_t j, uint32_t nrec, uint32_t top_pos) {
    extern __shared__ unsigned long long smask[];
    struct Wave {
        uint2 xyz[64];
        uint32_t mI[64], mB[64];
        uint16_t wl[26 * 64];
    };
    __shared__ Wave sw[GM_BLOCK / 64];
    __shared__ uint32_t sh[GM_BLOCK / 64][3];
    if (blockIdx.x < nrec) {
        recycle_blocks(d, P, j, blockIdx.x, nrec, smask);
        return;
    }
    const uint32_t halt = d.st->halt, nfull = d.win->full[j], csz = d.win->step[j].csz;
    if (halt) return;
    const uint32_t w = threadIdx.x >> 6, lane = threadIdx.x & 63u, blk = blockIdx.x - nrec;
    const uint32_t nch = (nfull + csz - 1u) / csz, cpd = (nch + P.nbd - 1u) / P.nbd;
    const uint32_t c0 = blk * cpd, c1 = c0 + cpd < nch ? c0 + cpd : nch;
    Wave &W = sw[w];
    uint32_t tI = 0, tB = 0, ntop = 0;
    bool wrapped = false;
    for (uint32_t c = c0 + w; c < c1; c += GM_BLOCK / 64u) {
        const uint32_t p = c * csz + lane;
        const bool valid = lane < csz && p < nfull;
        const uint32_t am = valid ? d.pmA[p] : 0u;
        const uint4 q0 = valid ? par_plane(d, GM_PAR1_CELL)[p] : make_uint4(0u, 0u, 0u, 0u);
        W.xyz[lane] = make_uint2(q0.x, q0.y);
        retire(d, q0.z, q0.w, valid, blk & (GM_SUBS - 1u));
        /* where the parent's grain stands in the order of rho: the one that sets
         * rhomax is counted, one before it (all without cells) has its count wrap */
        const uint32_t rp = valid ? d.rpos[q0.z] : 0xFFFFFFFFu;
        W.mI[lane] = 0;
        W.mB[lane] = 0;
        const uint32_t n = list_attempts(am, W.wl);
        for (uint32_t i = lane; i < n; i += 64u) {
            const uint32_t e = W.wl[i], q = e & 0xFFu, rk = e >> 8;
            const uint2 v = W.xyz[q];
            uint32_t tx, ty, tz;
            bool toB;
            attempt_target(d, (v.y >> 16) != 0u, v.x & 0xFFFFu, v.x >> 16, v.y & 0xFFFFu, (int)rk, tx, ty, tz, toB);
            const uint2 t = d.cell[cell_of(d, tx, ty, tz)];
            if (t.x == (c * csz + q) * 32u + rk) atomicOr(toB ? &W.mB[q] : &W.mI[q], 1u << rk);
            if (i < GM_GATT && c < d.gchunks) d.gatt[(size_t)c * GM_GATT + i] = t.y;
        }
        ntop += rp == top_pos ? 1u : 0u;
        wrapped |= rp < top_pos;
        wave_sync();
        const uint32_t mI = W.mI[lane], mB = W.mB[lane];
        if (valid) {
            d.pmI[p] = mI;
            d.pmB[p] = mB;
        }
        uint32_t cnt = (uint32_t)__popc(mI) << 16 | (uint32_t)__popc(mB);
        for (int o = 32; o > 0; o >>= 1) cnt += (uint32_t)__shfl_xor((int)cnt, o, 64);
        if (lane == 0) {
            d.ccnt[c] = cnt;
            tI += cnt >> 16;
            tB += cnt & 0xFFFFu;
        }
        wave_sync();
    }
    if (__any(wrapped) && lane == 0) d.st->cwrap = 1u;
    block_sum3(tI, tB, ntop, sh);
    if (threadIdx.x == 0) {
        d.btot[blk] = make_uint2(tI, tB);
        d.btop[blk] = ntop;
    }
}

/* New records as omp_infect_OutOfRXFront* write them (SCORE_Kernel.cpp:4281-4310,
 * :4402-4426), slots as omp_getNextFreeSlotIn* hand them out (:3757-3874).  A wave takes a chunk of
 * parents at a time; their winners are flattened into a list so that every lane
 * commits one infection.  Each lane loads its own parent's data with its winner
 * masks and shares it through LDS, and a winner issues its target's grain and its
 * slot lookup together, so a wave waits on few dependent memory round trips.
 * A winner's rank in its list is the winners before it: the blocks of the decide
 * pass before its own (added up by the block), the chunks before its own in that
 * block, the parents before its own in the chunk. */
static __device__ __forceinline__ void commit_step(const GmDev &d, const GmPParams &pp, const GmSweepArgs &A, const GmPart &P,
                                                   uint32_t j, uint32_t need_one) {
    struct Wave {
        uint32_t sA[64], sI[64], sB[64], oA[64], oI[64], oB[64];
        uint4 sq0[64];
        double sfin[64], sP[64];
        uint16_t wl[26 * 64];
    };
    __shared__ Wave sw[GM_BLOCK / 64];
    __shared__ uint32_t sh[GM_BLOCK / 64][3];
    GmStats *st = d.st;
    const uint32_t halt = st->halt, nfull = d.win->full[j];
    const GmWinStep ws = d.win->step[j];
    if (halt) return;
    const uint32_t k = A.k, csz = ws.csz;
    const uint32_t nch = (nfull + csz - 1u) / csz, cpd = (nch + P.nbd - 1u) / P.nbd, db = blockIdx.x;
    const uint32_t c0 = db * cpd, c1 = c0 + cpd < nch ? c0 + cpd : nch;
    if (c0 >= nch) return;
    const uint32_t lane = threadIdx.x & 63u, wv = threadIdx.x >> 6;
    /* a lane's parent: winner masks | x | y, z | fromB, defg, rxg | fin, P; the
     * wave's first chunk is loaded before the winners of earlier blocks are added up */
    uint32_t am, mI, mB;
    uint4 q0;
    double2 fp;
    auto load = [&](uint32_t c) {
        const uint32_t pt = c * csz + lane;
        am = mI = mB = 0;
        q0 = make_uint4(0u, 0u, 0xFFFFFFFFu, 0xFFFFFFFFu);
        fp = make_double2(0.0, 0.0);
        if (c < c1 && lane < csz && pt < nfull) {
            am = d.pmA[pt];
            mI = d.pmI[pt];
            mB = d.pmB[pt];
            q0 = par_plane(d, GM_PAR1_CELL)[pt];
            fp = reinterpret_cast<const double2 *>(par_plane(d, GM_PAR1_FP))[pt];
        }
    };
    load(c0 + wv);
    /* winners of the block's chunks [a, b) */
    auto count = [&](uint32_t a, uint32_t b, uint32_t &nI, uint32_t &nB) {
        nI = nB = 0;
        for (uint32_t i = a + lane; i < b; i += 64u) {
            const uint32_t v = d.ccnt[i];
            nI += v >> 16;
            nB += v & 0xFFFFu;
        }
    };
    uint32_t runI = 0, runB = 0, totI = 0;
    uint2 bt[4];
    static_assert(GM_DB <= 4 * GM_BLOCK, "one round of loads");
#pragma unroll
    for (uint32_t i = 0; i < 4u; i++) {
        const uint32_t at = threadIdx.x + i * GM_BLOCK;
        bt[i] = at < P.nbd ? d.btot[at] : make_uint2(0u, 0u);
    }
    uint32_t bI, bB;
    count(c0, c0 + wv < c1 ? c0 + wv : c1, bI, bB);
#pragma unroll
    for (uint32_t i = 0; i < 4u; i++) {
        const bool before = threadIdx.x + i * GM_BLOCK < db;
        totI += bt[i].x;
        runI += before ? bt[i].x : 0u;
        runB += before ? bt[i].y : 0u;
    }
    block_sum3(runI, runB, totI, sh);
    /* every block finds the same: the Inside list must grow before the step's
     * records go in, and the pass runs again */
    const uint64_t need = (uint64_t)ws.nI + (totI > ws.recLenI ? totI - ws.recLenI : 0u);
    if (need > d.capI && d.capI < d.capImax) {
        if (db == 0 && threadIdx.x == 0) {
            /* not st->halt, which the pass's other blocks read: two waves of one must
             * not see different values of it; the next propose pass halts on this */
            agent_store(&st->grow, need < d.capImax ? (uint32_t)need : d.capImax);
        }
        return;
    }
    Wave &W = sw[wv];
    bool one = false;
    for (uint32_t c = c0 + wv; c < c1; c += GM_BLOCK / 64u) {
        if (c != c0 + wv) {
            load(c);
            count(c - GM_BLOCK / 64u, c, bI, bB);
        }
        for (int o = 32; o > 0; o >>= 1) {
            bI += __shfl_xor(bI, o, 64);
            bB += __shfl_xor(bB, o, 64);
        }
        runI += bI;
        runB += bB;
        const uint32_t cI = (uint32_t)__popc(mI), cB = (uint32_t)__popc(mB);
        /* one scan of both counts (each batch total < 2^16) */
        const uint32_t packed = (cI << 16) | cB;
        const uint32_t incl = wave_incl_scan(packed);
        const uint32_t ex = incl - packed, tot = __shfl(incl, 63, 64);
        const uint32_t totI = tot >> 16, totB = tot & 0xFFFFu;
        const uint32_t na = (uint32_t)__popc(am);
        W.sA[lane] = am;
        W.oA[lane] = wave_incl_scan(na) - na;
        W.oI[lane] = runI + (ex >> 16);
        W.oB[lane] = runB + (ex & 0xFFFFu);
        W.sI[lane] = mI;
        W.sB[lane] = mB;
        W.sq0[lane] = q0;
        W.sfin[lane] = fp.x;
        W.sP[lane] = fp.y;
        /* winners of this parent at [exI + exB, ...) in the flat list, by rank */
        uint32_t pos = (ex >> 16) + (ex & 0xFFFFu);
        for (uint32_t m = mI | mB; m; m &= m - 1u) W.wl[pos++] = (uint16_t)(lane | ((uint32_t)__ffs(m) - 1u) << 8);
        wave_sync();
        const uint32_t nw = totI + totB;
        for (uint32_t w = lane; w < nw; w += 64u) {
            const uint32_t e = W.wl[w], q = e & 0xFFu, r = e >> 8, bit = 1u << r;
            const uint4 pq0 = W.sq0[q];
            uint32_t tx, ty, tz;
            bool toB;
            attempt_target(d, (pq0.y >> 16) != 0u, pq0.x & 0xFFFFu, pq0.x >> 16, pq0.y & 0xFFFFu, (int)r, tx, ty, tz,
                           toB);
            const uint32_t t = cell_of(d, tx, ty, tz);
            /* the target's grain, from the decide pass */
            const uint32_t ia = W.oA[q] + (uint32_t)__popc(W.sA[q] & (bit - 1u));
            const uint32_t g = ia < GM_GATT && c < d.gchunks ? d.gatt[(size_t)c * GM_GATT + ia] : d.cell[t].y;
            /* rank k into a list takes its k-th recycled slot, else appends */
            const uint32_t wI = W.sI[q];
            const bool intoI = (wI & bit) != 0u;
            const uint32_t wm = intoI ? wI : W.sB[q];
            const uint32_t rank = (intoI ? W.oI[q] : W.oB[q]) + (uint32_t)__popc(wm & (bit - 1u));
            const uint32_t recLen = intoI ? ws.recLenI : ws.recLenB;
            const uint32_t *recl = intoI ? d.recI : d.recB;
            const uint32_t rel = rank < recLen ? recl[rank] : (intoI ? ws.nI : ws.nB) + (rank - recLen);
            const NewCell nc = new_cell(d, pp, A, k, W.sfin[q], W.sP[q], pq0, r, g);
            one |= nc.one;
            if (rel >= (intoI ? d.capI : d.capB)) {
                atomicOr(&st->err, intoI ? GM_ERRF_INSIDE_FULL : GM_ERRF_BORDER_FULL);
                continue;
            }
            put_cell(d, k, nc, pq0, t, g, tx, ty, tz, intoI ? d.baseI + rel : rel);
        }
        wave_sync();
    }
    /* (stores to one address are served one after another: only where it matters) */
    if (need_one && __any(one) && lane == 0) agent_store(&st->pone, 1u);
}

static __device__ void window_end(const GmDev &d, const GmPart &P, uint32_t launched, uint32_t top_pos, uint32_t *out);

/* the cells left of the grain that sets rhomax after step j, by the pass's last block,
 * which most often has no parents (and in a pass that runs again finds the same) */
static __device__ __forceinline__ void count_top(const GmDev &d, const GmPart &P, uint32_t j) {
    __shared__ uint32_t sh[GM_BLOCK / 64][3];
    const uint32_t halt = d.st->halt, had = d.win->left[j];
    uint32_t n = 0, z0 = 0, z1 = 0;
    for (uint32_t i = threadIdx.x; i < P.nbd; i += GM_BLOCK) n += d.btop[i];
    if (halt) return;
    block_sum3(n, z0, z1, sh);
    if (threadIdx.x == 0) {
        d.win->left[j + 1u] = had - n;
        if (n && had == n) agent_store(&d.win->top_hit, 1u);
    }
}

/* With `out` the pass is the window's last: the block that finds all others done closes
 * the window (window_end), where a launch of its own took 6 us a window: a tenth of a
 * step where the scalars change in every one.  What it needs of the other
 * blocks they change by device atomics alone (counters, flags, the new pairs' keys),
 * so no block has to write its XCD's cache back; each waits until its own have
 * arrived before it takes its ticket. */
__global__ void __launch_bounds__(GM_BLOCK, 4) k_commit(GmDev d, GmPParams pp, GmSweepArgs A, GmPart P, uint32_t j,
                                                       uint32_t need_one, uint32_t top_pos, uint32_t *out) {
    __shared__ uint32_t last;
    commit_step(d, pp, A, P, j, need_one);
    if (blockIdx.x == gridDim.x - 1u) count_top(d, P, j);
    if (!out) return;
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (threadIdx.x == 0) last = atomicAdd(&d.st->ticket, 1u) == gridDim.x - 1u ? 1u : 0u;
    __syncthreads();
    if (last) window_end(d, P, j + 1u, top_pos, out);
}

hipError_t gm_launch_infect(const GmDev &d, const GmPParams &pp, const GmSweepArgs &a, const GmPart &P,
                            const GmWindow &w, uint32_t j, GmStats *out, hipStream_t s, hipEvent_t *ev) {
    hipError_t e;
    if ((e = mark(ev, 4, s)) != hipSuccess) return e;
    if (j || !P.fused) k_propose<<<P.nbp + 1u, GM_BLOCK, 0, s>>>(d, P, w, j, a.k + j);
    if ((e = mark(ev, 5, s)) != hipSuccess) return e;
    const uint32_t nrec = P.nb < GM_RECYCLE_BLOCKS ? P.nb : GM_RECYCLE_BLOCKS;
    /* a sweep block's INACTIVE masks and the offsets of its tiles */
    const size_t lds = (size_t)GM_SW_WAVES * P.cpw * GM_SW_TPC * (sizeof(unsigned long long) + sizeof(uint32_t));
    k_decide<<<nrec + P.nbd, GM_BLOCK, lds, s>>>(d, P, j, nrec, w.top_pos);
    for (int i = 6; i <= 8; i++)
        if ((e = mark(ev, i, s)) != hipSuccess) return e;
    return gm_launch_commit(d, pp, a, P, w, j, out, s, ev);
}

hipError_t gm_launch_commit(const GmDev &d, const GmPParams &pp, const GmSweepArgs &a, const GmPart &P,
                            const GmWindow &w, uint32_t j, GmStats *out, hipStream_t s, hipEvent_t *ev) {
    hipError_t e;
    GmSweepArgs A = a;
    A.k = a.k + j;
    k_commit<<<P.nbd, GM_BLOCK, 0, s>>>(d, pp, A, P, j, w.need_one, w.top_pos, reinterpret_cast<uint32_t *>(out));
    if ((e = mark(ev, 9, s)) != hipSuccess) return e;
    return hipGetLastError();
}

/* what the decide pass of step j retired, back (the parts of a count are only ever added up) */
__global__ void k_unretire(GmDev d, uint32_t j) {
    const uint32_t nfull = d.win->full[j];
    for (uint32_t p = blockIdx.x * blockDim.x + threadIdx.x; p < nfull; p += gridDim.x * blockDim.x) {
        const uint4 q = par_plane(d, GM_PAR1_CELL)[p];
        atomicSub(&d.defsub[q.z], 1u);
        atomicSub(&d.rxcnt[q.w], 1u);
    }
}

hipError_t gm_launch_unretire(const GmDev &d, uint32_t j, hipStream_t s) {
    k_unretire<<<GM_DB, GM_BLOCK, 0, s>>>(d, j);
    return hipGetLastError();
}

/* exported map, SCORE's raw file encoding: 1 for an infected cell, else 2 + id */
__global__ void k_raw2gid(uint32_t *m, uint64_t n) {
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x)
        m[i] = m[i] == GM_INFECTED ? 1u : 2u + m[i];
}

hipError_t gm_launch_raw2gid(uint32_t *m, uint64_t n, hipStream_t s) {
    k_raw2gid<<<fill_blocks(n), GM_BLOCK, 0, s>>>(m, n);
    return hipGetLastError();
}

/* exported map: the grains the cells came with */
__global__ void k_grid_out(GmDev d, uint32_t *out) {
    const uint32_t n2 = (uint32_t)(d.N / 2u);
    const uint4 *in = reinterpret_cast<const uint4 *>(d.cell);
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n2; i += gridDim.x * blockDim.x) {
        const uint4 q = in[i];
        reinterpret_cast<uint2 *>(out)[i] = make_uint2(q.y, q.w);
    }
    if ((d.N & 1u) && blockIdx.x == 0 && threadIdx.x == 0) out[d.N - 1u] = d.cell[d.N - 1u].y;
}

/* exported map: retired cells from the log (a cell retired twice is its nucleus' both
 * times) */
__global__ void k_apply_rlog(GmDev d, uint32_t *out) {
    const unsigned long long n = d.st->nret < d.rlogCap ? d.st->nret : d.rlogCap;
    for (unsigned long long i = (unsigned long long)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (unsigned long long)gridDim.x * blockDim.x) {
        const uint2 e = d.rlog[i];
        out[e.x] = e.y;
    }
}

/* exported map: cells held by active front records before step k are INFECTED */
__global__ void k_overlay_infected(GmDev d, uint32_t nI, uint32_t nB, uint32_t k, uint32_t *out) {
    const uint32_t n = nI + nB, kc = k & (GM_CS_MOD - 1u);
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const uint32_t s = occ_slot(d, nI, i);
        if (!cs_inactive(d.cstep[s], kc, d.horizon)) out[d.rec[s].cell] = GM_INFECTED;
    }
}

hipError_t gm_launch_overlay_infected(const GmDev &d, uint32_t nI, uint32_t nB, uint32_t k, uint32_t *out,
                                      hipStream_t s) {
    k_grid_out<<<fill_blocks((d.N + 1u) / 2u), GM_BLOCK, 0, s>>>(d, out);
    /* a cell is infected once, and retired after that: where another record still holds it
     * (a defragmentation took it back) SCORE's grid has the retirement */
    if (nI + nB) k_overlay_infected<<<fill_blocks(nI + nB), GM_BLOCK, 0, s>>>(d, nI, nB, k, out);
    k_apply_rlog<<<8192, GM_BLOCK, 0, s>>>(d, out);
    return hipGetLastError();
}

/* ------------------------------------------------- device-wide exclusive scan
 * (nucleation only) Two u32 arrays scanned in place over n entries.  Fixed grid:
 * block b owns a contiguous chunk; phase 2 scans the block sums. */

static __device__ __forceinline__ uint32_t block_incl_scan(uint32_t v, uint32_t *total) {
    __shared__ uint32_t ws[GM_BLOCK / 64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    uint32_t inc = wave_incl_scan(v);
    if (lane == 63) ws[w] = inc;
    __syncthreads();
    uint32_t pre = 0, tot = 0;
#pragma unroll
    for (int i = 0; i < GM_BLOCK / 64; i++) {
        uint32_t x = ws[i];
        if (i < w) pre += x;
        tot += x;
    }
    __syncthreads();
    *total = tot;
    return inc + pre;
}

static __device__ __forceinline__ void chunk_of(uint32_t n, uint32_t &lo, uint32_t &hi) {
    uint32_t per = (n + gridDim.x - 1) / gridDim.x;
    per = (per + GM_BLOCK - 1) / GM_BLOCK * GM_BLOCK;
    lo = blockIdx.x * per;
    hi = lo + per;
    if (lo > n) lo = n;
    if (hi > n) hi = n;
}

__global__ void k_scan_p1(const uint32_t *a, const uint32_t *b, uint32_t n, uint32_t *bsum) {
    uint32_t lo, hi;
    chunk_of(n, lo, hi);
    uint32_t sa = 0, sb = 0;
    for (uint32_t i = lo + threadIdx.x; i < hi; i += GM_BLOCK) {
        sa += a[i];
        sb += b[i];
    }
    uint32_t ta, tb;
    block_incl_scan(sa, &ta);
    block_incl_scan(sb, &tb);
    if (threadIdx.x == 0) {
        bsum[blockIdx.x] = ta;
        bsum[gridDim.x + blockIdx.x] = tb;
    }
}

__global__ void k_scan_p2(uint32_t *bsum, uint32_t nb, uint32_t *totals) {
    __shared__ uint32_t wsa[16], wsb[16];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    uint32_t va = threadIdx.x < nb ? bsum[threadIdx.x] : 0u;
    uint32_t vb = threadIdx.x < nb ? bsum[nb + threadIdx.x] : 0u;
    uint32_t ia = wave_incl_scan(va), ib = wave_incl_scan(vb);
    if (lane == 63) { wsa[w] = ia; wsb[w] = ib; }
    __syncthreads();
    uint32_t pa = 0, pb = 0, ta = 0, tb = 0;
    for (int i = 0; i < 16; i++) {
        if (i < w) { pa += wsa[i]; pb += wsb[i]; }
        ta += wsa[i];
        tb += wsb[i];
    }
    if (threadIdx.x < nb) {
        bsum[threadIdx.x] = ia - va + pa;
        bsum[nb + threadIdx.x] = ib - vb + pb;
    }
    if (threadIdx.x == 0) { totals[0] = ta; totals[1] = tb; }
}

__global__ void k_scan_p3(uint32_t *a, uint32_t *b, uint32_t n, const uint32_t *bsum) {
    uint32_t lo, hi;
    chunk_of(n, lo, hi);
    uint32_t ra = bsum[blockIdx.x], rb = bsum[gridDim.x + blockIdx.x];
    for (uint32_t base = lo; base < hi; base += GM_BLOCK) {
        uint32_t i = base + threadIdx.x;
        uint32_t va = i < hi ? a[i] : 0u, vb = i < hi ? b[i] : 0u;
        uint32_t ta, tb;
        uint32_t ia = block_incl_scan(va, &ta);
        uint32_t ib = block_incl_scan(vb, &tb);
        if (i < hi) {
            a[i] = ra + ia - va;
            b[i] = rb + ib - vb;
        }
        ra += ta;
        rb += tb;
    }
}

static hipError_t scan2(const GmDev &d, uint32_t *a, uint32_t *b, uint32_t n, hipStream_t s) {
    uint32_t nb = (n + GM_BLOCK - 1) / GM_BLOCK;
    if (nb > GM_SCAN_BLOCKS) nb = GM_SCAN_BLOCKS;
    if (nb < 1) nb = 1;
    k_scan_p1<<<nb, GM_BLOCK, 0, s>>>(a, b, n, d.scan_bsum);
    k_scan_p2<<<1, 1024, 0, s>>>(d.scan_bsum, nb, d.st->scan_tot);
    k_scan_p3<<<nb, GM_BLOCK, 0, s>>>(a, b, n, d.scan_bsum);
    return hipGetLastError();
}

/* ------------------------------------------------------------ nucleation
 * ompshar_sim_myCA_sitesaturatedNucleation + infect_JuvenileNucleation
 * (SCORE_GrowthMachine.cpp:50-189): nuclei in pool order, a site already taken
 * rejects later nuclei; interior sites append to Inside, shell sites to Border. */

static __device__ __forceinline__ bool site_deformed(const GmDev &d, uint32_t w) {
    const uint32_t z = w / d.nxy, rem = w - z * d.nxy, y = rem / d.nx, x = rem - y * d.nx;
    return is_deformed(d, x, y, z);
}

__global__ void k_nuc_claim(GmDev d, const uint32_t *site, uint32_t n) {
    for (uint32_t k = blockIdx.x * blockDim.x + threadIdx.x; k < n; k += gridDim.x * blockDim.x) {
        uint32_t w = site[k];
        if (w != GM_NO_SITE && site_deformed(d, w)) atomicMin(&d.cell[w].x, k);
    }
}

static __device__ __forceinline__ bool site_interior(const GmDev &d, uint32_t w) {
    uint32_t z = w / d.nxy, rem = w - z * d.nxy, y = rem / d.nx, x = rem - y * d.nx;
    return x > 0 && x < d.nx - 1 && y > 0 && y < d.ny - 1 && z > 0 && z < d.nz - 1;
}

__global__ void k_nuc_flag(GmDev d, const uint32_t *site, uint32_t n) {
    for (uint32_t k = blockIdx.x * blockDim.x + threadIdx.x; k < n; k += gridDim.x * blockDim.x) {
        uint32_t w = site[k];
        bool win = w != GM_NO_SITE && site_deformed(d, w) && d.cell[w].x == k;
        bool in = win && site_interior(d, w);
        d.nI_[k] = (win && in) ? 1u : 0u;
        d.nB_[k] = (win && !in) ? 1u : 0u;
        d.nflag[k] = win ? 1u : 0u;
    }
}

__global__ void k_nuc_commit(GmDev d, const uint32_t *site, const double *nucP, uint32_t n) {
    for (uint32_t k = blockIdx.x * blockDim.x + threadIdx.x; k < n; k += gridDim.x * blockDim.x) {
        if (!d.nflag[k]) continue;
        uint32_t w = site[k];
        bool in = site_interior(d, w);
        uint32_t gslot;
        if (in) {
            gslot = d.nI_[k];
            if (gslot >= d.capI) { atomicOr(&d.st->err, GM_ERRF_INSIDE_FULL); continue; }
            gslot += d.baseI;
        } else {
            uint32_t rel = d.nB_[k];
            if (rel >= d.capB) { atomicOr(&d.st->err, GM_ERRF_BORDER_FULL); continue; }
            gslot = rel;
        }
        uint32_t g = d.cell[w].y;
        GmRec *r = d.rec + gslot;
        rec_set_a(r, 1.0, 0u, 26u);
        rec_set_b(r, 0.0);
        rec_set_c(r, nucP[k], w, g);
        r->rxg = k;
        d.cstep[gslot] = (gm_cs_t)GM_CS_UNKNOWN;
        const uint32_t z = w / d.nxy, rem = w - z * d.nxy, y = rem / d.nx, x = rem - y * d.nx;
        clear_deformed(d, x, y, z);
    }
}

__global__ void k_nuc_tail(GmDev d) {
    d.st->nI = d.st->scan_tot[0];
    d.st->nB = d.st->scan_tot[1];
    if (d.st->nB > d.capB) atomicOr(&d.st->err, GM_ERRF_BORDER_FULL);
}

hipError_t gm_launch_nucleate(const GmDev &d, const uint32_t *site, const double *nucP, uint32_t n, hipStream_t s) {
    if (n == 0) {
        k_fill_u32<<<1, 32, 0, s>>>(d.st->scan_tot, 0u, 2);
        k_nuc_tail<<<1, 1, 0, s>>>(d);
        return hipGetLastError();
    }
    unsigned nb = fill_blocks(n);
    k_nuc_claim<<<nb, GM_BLOCK, 0, s>>>(d, site, n);
    k_nuc_flag<<<nb, GM_BLOCK, 0, s>>>(d, site, n);
    hipError_t e = scan2(d, d.nI_, d.nB_, n, s);
    if (e != hipSuccess) return e;
    k_nuc_commit<<<nb, GM_BLOCK, 0, s>>>(d, site, nucP, n);
    k_nuc_tail<<<1, 1, 0, s>>>(d);
    return hipGetLastError();
}

/* ------------------------------------------------------ mobility-weight cache */

__global__ void k_resolve_pending(GmDev d, const double *vals, uint32_t n) {
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
        d.hvals[d.pend_slot[i]] = vals[i];
}

hipError_t gm_launch_resolve_pending(const GmDev &d, const double *vals, uint32_t n, hipStream_t s) {
    if (n == 0) return hipSuccess;
    k_resolve_pending<<<fill_blocks(n), GM_BLOCK, 0, s>>>(d, vals, n);
    return hipGetLastError();
}

__global__ void __launch_bounds__(GM_BLOCK) k_stats_out(GmDev d, uint32_t *out) { copy_stats(d, out); }

hipError_t gm_launch_stats_out(const GmDev &d, GmStats *out, hipStream_t s) {
    k_stats_out<<<1, GM_BLOCK, 0, s>>>(d, reinterpret_cast<uint32_t *>(out));
    return hipGetLastError();
}

/* The end of a window of `launched` steps, by one block: its last step is closed,
 * unless the window halted (the propose pass that halted it closed the step before),
 * and the stats go to the host. */
static __device__ void window_end(const GmDev &d, const GmPart &P, uint32_t launched, uint32_t top_pos, uint32_t *out) {
    if (!d.st->halt && !agent_load(&d.st->grow) && d.st->nexec + 1u == launched) close_step(d, P, launched - 1u, false);
    stats_to_host(d, top_pos, out);
}

__global__ void __launch_bounds__(GM_BLOCK) k_window_end(GmDev d, GmPart P, uint32_t launched, uint32_t top_pos,
                                                         uint32_t *out) {
    window_end(d, P, launched, top_pos, out);
}

hipError_t gm_launch_window_end(const GmDev &d, const GmPart &P, uint32_t launched, uint32_t top_pos, GmStats *out,
                                hipStream_t s) {
    k_window_end<<<1, GM_BLOCK, 0, s>>>(d, P, launched, top_pos, reinterpret_cast<uint32_t *>(out));
    return hipGetLastError();
}

/* SCORE's per-slot view before step k: activity, rxFrac (replayed from the
 * anchor; INACTIVE slots hold 0.0 as the reference leaves them), and the record
 * fields, with pending weights replaced by their cached values in the record
 * itself.  With o.act null only the weights are resolved. */
__global__ void k_materialize(GmDev d, uint32_t k, uint32_t base, uint32_t n, GmFrontOut o) {
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const uint32_t s = base + i;
        const uint32_t cs = d.cstep[s];
        GmRec *r = d.rec + s;
        const RecA a = rec_a(r);
        const RecC c = rec_c(r);
        const double P = resolved(d, c.P);
        if (is_pending(c.P)) r->P = P;
        if (!o.act) continue;
        o.P[i] = P;
        o.inf[i] = (uint8_t)a.inf;
        o.cell[i] = c.cell;
        o.defg[i] = c.defg;
        o.rxg[i] = r->rxg;
        if (cs_inactive(cs, k & (GM_CS_MOD - 1u), d.horizon)) {
            o.act[i] = 0;
            o.frac[i] = 0.0;
            continue;
        }
        o.act[i] = 1;
        double f = a.frac0;
        if (cs != GM_CS_UNKNOWN) f = gm_radd_n(f, r->inc, k - a.s0);
        o.frac[i] = f;
    }
}

hipError_t gm_launch_materialize(const GmDev &d, uint32_t k, uint32_t base, uint32_t n, const GmFrontOut &o,
                                 hipStream_t s) {
    if (n == 0) return hipSuccess;
    k_materialize<<<fill_blocks(n), GM_BLOCK, 0, s>>>(d, k, base, n, o);
    return hipGetLastError();
}

__global__ void k_hash_insert(GmDev d, const unsigned long long *keys, const double *vals, uint32_t n) {
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        unsigned long long key = keys[i];
        uint32_t h = hash_slot(key, d.hcap);
        const uint32_t nprobe = d.hcap < GM_PROBE_MAX ? d.hcap : GM_PROBE_MAX;
        bool stored = false;
        for (uint32_t probe = 0; probe < nprobe; probe++) {
            unsigned long long old = atomicCAS(&d.hkeys[h], 0ull, key);
            if (old == 0ull || old == key) {
                d.hvals[h] = vals[i];
                stored = true;
                break;
            }
            h = (h + 1u) & (d.hcap - 1u);
        }
        /* lookups stop after nprobe slots, so a key stored further away would be
         * lost; the host grows the table and inserts again */
        if (!stored) atomicOr(&d.st->err, GM_ERRF_PCACHE_FULL);
    }
}

hipError_t gm_launch_hash_insert(const GmDev &d, const unsigned long long *keys, const double *vals, uint32_t n,
                                 hipStream_t s) {
    if (n == 0) return hipSuccess;
    k_hash_insert<<<fill_blocks(n), GM_BLOCK, 0, s>>>(d, keys, vals, n);
    return hipGetLastError();
}

/* ------------------------------------------------------- defragmentation
 * ompshar_defragmentation (SCORE_Kernel.cpp:3877-3934), one list at a time: the
 * first INACTIVE slot is found (past nextSlotNeverActive if every slot below it
 * is ACTIVE, as the reference's unbounded search does), then every ACTIVE slot
 * after it moves down, in order, to close the gaps.  The reference copies the
 * records and leaves the slots behind the compacted block as they were; an
 * ACTIVE record left there is frozen here at its value before step k (anchor k,
 * increment 0), which is what the reference holds in that slot from then on. */

__global__ void __launch_bounds__(GM_BLOCK) k_defrag_first(GmDev d, uint32_t base, uint32_t lo, uint32_t hi,
                                                          uint32_t kc) {
    const uint32_t lane = threadIdx.x & 63u, stride = gridDim.x * GM_BLOCK;
    for (uint32_t i0 = lo + blockIdx.x * GM_BLOCK + (threadIdx.x & ~63u); i0 < hi; i0 += stride) {
        const uint32_t i = i0 + lane;
        const uint64_t m = __ballot(i < hi && cs_inactive(d.cstep[base + i], kc, d.horizon));
        if (m) {
            /* later chunks of this wave only hold larger slots */
            if (lane == 0) atomicMin(&d.st->dfirst, i0 + (uint32_t)__ffsll((long long)m) - 1u);
            return;
        }
        if (hi - i0 <= stride) return;
    }
}

hipError_t gm_launch_defrag_first_inactive(const GmDev &d, uint32_t base, uint32_t lo, uint32_t hi, uint32_t k,
                                           hipStream_t s) {
    k_fill_u32<<<1, 64, 0, s>>>(&d.st->dfirst, hi, 1);
    if (hi > lo) k_defrag_first<<<fill_blocks(hi - lo), GM_BLOCK, 0, s>>>(d, base, lo, hi, k & (GM_CS_MOD - 1u));
    return hipGetLastError();
}

/* ACTIVE slots among list slots first+1+i, i in [0, n), per block chunk */
__global__ void __launch_bounds__(GM_BLOCK) k_defrag_count(GmDev d, uint32_t base, uint32_t first, uint32_t n,
                                                          uint32_t kc) {
    uint32_t lo, hi;
    chunk_of(n, lo, hi);
    uint32_t c = 0;
    for (uint32_t i = lo + threadIdx.x; i < hi; i += GM_BLOCK)
        c += cs_inactive(d.cstep[base + first + 1u + i], kc, d.horizon) ? 0u : 1u;
    uint32_t tot;
    block_incl_scan(c, &tot);
    if (threadIdx.x == 0) d.bcnt[blockIdx.x] = tot;
}

/* exclusive scan of one row of per-block counts; the total goes to st->dcount */
__global__ void __launch_bounds__(1024) k_scan_row(GmDev d, uint32_t nb) {
    uint32_t tot[1];
    scan_block_counts<1>(d.bcnt, nb, tot);
    if (threadIdx.x == 0) d.st->dcount = tot[0];
}

/* Each ACTIVE record after `first` is copied, in slot order, to the scratch
 * array; one that the compacted block will not overwrite is then frozen. */
__global__ void __launch_bounds__(GM_BLOCK) k_defrag_gather(GmDev d, uint32_t base, uint32_t first, uint32_t n,
                                                           uint32_t k, GmRec *trec, gm_cs_t *tcs) {
    uint32_t lo, hi;
    chunk_of(n, lo, hi);
    uint32_t run = d.bcnt[blockIdx.x];
    const uint32_t keep = first + d.st->dcount; /* list slots below this receive moved records */
    for (uint32_t b0 = lo; b0 < hi; b0 += GM_BLOCK) {
        const uint32_t i = b0 + threadIdx.x;
        const uint32_t c = first + 1u + i;
        const uint32_t cs = i < hi ? d.cstep[base + c] : GM_CS_INACTIVE;
        const uint32_t act = cs_inactive(cs, k & (GM_CS_MOD - 1u), d.horizon) ? 0u : 1u;
        /* the code of a cell that completed in an earlier step becomes the
         * sentinel, so that no past code stays behind the compacted block */
        if (i < hi && !act && cs != GM_CS_INACTIVE) d.cstep[base + c] = (gm_cs_t)GM_CS_INACTIVE;
        uint32_t tot;
        const uint32_t incl = block_incl_scan(act, &tot);
        if (act) {
            const uint32_t o = run + incl - 1u;
            GmRec *r = d.rec + base + c;
            const uint4 *src = reinterpret_cast<const uint4 *>(r);
            const uint4 q0 = src[0], q1 = src[1], q2 = src[2], q3 = src[3];
            uint4 *dst = reinterpret_cast<uint4 *>(trec + o);
            dst[0] = q0;
            dst[1] = q1;
            dst[2] = q2;
            dst[3] = q3;
            tcs[o] = (gm_cs_t)cs;
            if (c >= keep) {
                double f = __hiloint2double((int)q0.y, (int)q0.x);
                const double inc = __hiloint2double((int)q1.y, (int)q1.x);
                if (cs != GM_CS_UNKNOWN) f = gm_radd_n(f, inc, k - q0.z);
                const double P = resolved(d, __hiloint2double((int)q2.y, (int)q2.x));
                rec_set_a(r, f, k, q0.w);
                rec_set_b(r, 0.0);
                rec_set_c(r, P, q2.z, q2.w);
                d.cstep[base + c] = (gm_cs_t)GM_CS_NEVER;
            }
        }
        run += tot;
    }
}

__global__ void __launch_bounds__(GM_BLOCK) k_defrag_scatter(GmDev d, uint32_t base, uint32_t first,
                                                            const GmRec *trec, const gm_cs_t *tcs) {
    const uint32_t n = d.st->dcount;
    for (uint32_t i = blockIdx.x * GM_BLOCK + threadIdx.x; i < n; i += gridDim.x * GM_BLOCK) {
        const uint4 *src = reinterpret_cast<const uint4 *>(trec + i);
        uint4 *dst = reinterpret_cast<uint4 *>(d.rec + base + first + i);
        const uint4 q0 = src[0], q1 = src[1], q2 = src[2], q3 = src[3];
        dst[0] = q0;
        dst[1] = q1;
        dst[2] = q2;
        dst[3] = q3;
        d.cstep[base + first + i] = tcs[i];
    }
}

hipError_t gm_launch_defrag_move(const GmDev &d, uint32_t base, uint32_t first, uint32_t nnever, uint32_t k,
                                 GmRec *trec, gm_cs_t *tcs, hipStream_t s) {
    if (first + 1u >= nnever) return hipSuccess;
    const uint32_t n = nnever - first - 1u;
    const uint32_t nb = grid_for(n, 4 * GM_BLOCK);
    k_defrag_count<<<nb, GM_BLOCK, 0, s>>>(d, base, first, n, k & (GM_CS_MOD - 1u));
    k_scan_row<<<1, 1024, 0, s>>>(d, nb);
    k_defrag_gather<<<nb, GM_BLOCK, 0, s>>>(d, base, first, n, k, trec, tcs);
    k_defrag_scatter<<<fill_blocks(n), GM_BLOCK, 0, s>>>(d, base, first, trec, tcs);
    return hipGetLastError();
}

/* ------------------------------------------------------------ status vector
 * ompcrit_clarify_status_infectedcells (SCORE_Io_Characterization.cpp:925-997):
 * every ACTIVE record, Inside list then Border list in slot order, as its
 * linear cell index and the grain the cell shows before step k: ndefg+rxg once
 * rxFrac has reached the threshold, else its deformed grain.  Item i of
 * [0, nI+nB) is Inside slot i or Border slot i-nI. */

static __device__ __forceinline__ uint32_t item_slot(const GmDev &d, uint32_t nI, uint32_t i) {
    return occ_slot(d, nI, i);
}

__global__ void __launch_bounds__(GM_BLOCK) k_status_count(GmDev d, uint32_t nI, uint32_t n, uint32_t kc) {
    uint32_t lo, hi;
    chunk_of(n, lo, hi);
    uint32_t c = 0;
    for (uint32_t i = lo + threadIdx.x; i < hi; i += GM_BLOCK)
        c += cs_inactive(d.cstep[item_slot(d, nI, i)], kc, d.horizon) ? 0u : 1u;
    uint32_t tot;
    block_incl_scan(c, &tot);
    if (threadIdx.x == 0) d.bcnt[blockIdx.x] = tot;
}

__global__ void __launch_bounds__(GM_BLOCK) k_status_write(GmDev d, uint32_t nI, uint32_t n, uint32_t k, double thr,
                                                          uint32_t *ixyz, uint32_t *gid) {
    uint32_t lo, hi;
    chunk_of(n, lo, hi);
    uint32_t run = d.bcnt[blockIdx.x];
    for (uint32_t b0 = lo; b0 < hi; b0 += GM_BLOCK) {
        const uint32_t i = b0 + threadIdx.x;
        const uint32_t s = i < hi ? item_slot(d, nI, i) : 0u;
        const uint32_t cs = i < hi ? d.cstep[s] : GM_CS_INACTIVE;
        const uint32_t act = cs_inactive(cs, k & (GM_CS_MOD - 1u), d.horizon) ? 0u : 1u;
        uint32_t tot;
        const uint32_t incl = block_incl_scan(act, &tot);
        if (act) {
            const GmRec *r = d.rec + s;
            const RecA a = rec_a(r);
            const RecC c = rec_c(r);
            double f = a.frac0;
            if (cs != GM_CS_UNKNOWN) f = gm_radd_n(f, r->inc, k - a.s0);
            const uint32_t o = run + incl - 1u;
            ixyz[o] = c.cell;
            gid[o] = f < thr ? c.defg : d.ndefg + r->rxg;
        }
        run += tot;
    }
}

hipError_t gm_launch_status(const GmDev &d, uint32_t nI, uint32_t nB, uint32_t k, double thr, uint32_t *ixyz,
                            uint32_t *gid, hipStream_t s) {
    const uint32_t n = nI + nB;
    if (n == 0) {
        k_fill_u32<<<1, 64, 0, s>>>(&d.st->dcount, 0u, 1);
        return hipGetLastError();
    }
    const uint32_t nb = grid_for(n, 4 * GM_BLOCK);
    k_status_count<<<nb, GM_BLOCK, 0, s>>>(d, nI, n, k & (GM_CS_MOD - 1u));
    k_scan_row<<<1, 1024, 0, s>>>(d, nb);
    k_status_write<<<nb, GM_BLOCK, 0, s>>>(d, nI, n, k, thr, ixyz, gid);
    return hipGetLastError();
}

/* ------------------------------------------------------------- arrivals
 * Nuclei that arrive after step 0 are placed at the start of their step, before
 * the sweep, as infect_JuvenileNucleation places the site-saturated ones
 * (SCORE_GrowthMachine.cpp:124-189): in pool order, a nucleus whose cell is no
 * longer deformed (taken by the front or by an earlier nucleus) is rejected;
 * the record (rxFrac 1.0, infector 26, the host's weight) is appended to the
 * Inside list for a strictly interior cell, else to the Border list.  The
 * reference marks this injection point but has no model behind it
 * (SCORE_Kernel.cpp:6632).  One block: every nucleus of the step claims its
 * cell (the lowest pool id wins), then the winners are ranked in pool order,
 * 1024 at a time, and each record is predicted under the step's scalars. */
__global__ void __launch_bounds__(1024) k_arrivals(GmDev d, GmSweepArgs A) {
    __shared__ uint32_t ws[16][2];
    GmStats *st = d.st;
    const uint32_t k = A.k; /* the first step of a window */
    if (k == 0u || k > d.arr_last) return;
    const uint32_t lo = d.arr_off[k], hi = d.arr_off[k + 1u];
    if (lo == hi) return;
    const uint32_t tid = threadIdx.x, lane = tid & 63u, w = tid >> 6;
    for (uint32_t i = lo + tid; i < hi; i += 1024u) {
        const uint32_t id = d.arr_ids[i], c = d.nsite[id];
        if (site_deformed(d, c)) atomicMin(&d.cell[c].x, id);
    }
    __syncthreads();
    uint32_t runI = st->nI, runB = st->nB, placed = 0;
    unsigned long long pk = 0ull;
    for (uint32_t base = lo; base < hi; base += 1024u) {
        const uint32_t i = base + tid;
        uint32_t id = 0, c = 0;
        bool win = false, in = false;
        if (i < hi) {
            id = d.arr_ids[i];
            c = d.nsite[id];
            win = site_deformed(d, c) &&
                  __hip_atomic_load(&d.cell[c].x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == id;
            in = win && site_interior(d, c);
        }
        const uint32_t vI = (win && in) ? 1u : 0u, vB = (win && !in) ? 1u : 0u;
        const uint32_t packed = (vI << 16) | vB;
        const uint32_t incl = wave_incl_scan(packed);
        if (lane == 63u) {
            ws[w][0] = incl >> 16;
            ws[w][1] = incl & 0xFFFFu;
        }
        __syncthreads();
        uint32_t preI = 0, preB = 0, totI = 0, totB = 0;
        for (uint32_t q = 0; q < 16u; q++) {
            if (q < w) { preI += ws[q][0]; preB += ws[q][1]; }
            totI += ws[q][0];
            totB += ws[q][1];
        }
        if (win) {
            const uint32_t ex = incl - packed;
            const uint32_t rel = in ? runI + preI + (ex >> 16) : runB + preB + (ex & 0xFFFFu);
            if (rel >= (in ? d.capI : d.capB)) {
                atomicOr(&st->err, in ? GM_ERRF_INSIDE_FULL : GM_ERRF_BORDER_FULL);
            } else {
                const uint32_t gslot = in ? d.baseI + rel : rel;
                const uint32_t g = d.cell[c].y;
                const double P = d.nucP[id];
                double inc = 0.0;
                const gm_cs_t cs = cs_code(d, predict_values(A, k, 1.0, P, d.rho[g], 26u, inc), k);
                GmRec *r = d.rec + gslot;
                rec_set_a(r, 1.0, k, 26u);
                rec_set_b(r, inc);
                rec_set_c(r, P, c, g);
                *reinterpret_cast<uint4 *>(&r->rxg) = make_uint4(id, 0u, 0u, 0u);
                d.cstep[gslot] = cs;
                const uint32_t z = c / d.nxy, rem = c - z * d.nxy, y = rem / d.nx, x = rem - y * d.nx;
                clear_deformed(d, x, y, z);
                const unsigned long long key = gm_pkey(P);
                pk = key > pk ? key : pk;
            }
        }
        runI += totI;
        runB += totB;
        placed += totI + totB;
        __syncthreads();
    }
    /* the block's largest weight */
    for (int o = 32; o > 0; o >>= 1) {
        const unsigned long long other = (unsigned long long)__shfl_down((long long)pk, o, 64);
        pk = other > pk ? other : pk;
    }
    if (lane == 0u && pk) atomicMax(&st->arr_pkey, pk);
    if (tid == 0) {
        st->nI = runI < d.capI ? runI : d.capI;
        st->nB = runB < d.capB ? runB : d.capB;
        st->nplaced = placed;
    }
}

/* ----------------------------------------------------------- launch windows
 * Up to GM_WMAX steps are launched back to back.  Every kernel of a step takes the
 * lists' lengths before it from the device (GmWin; with several regions the step's
 * index too, from the stats) and returns at once once a step has set `halt`, so that
 * the host takes over at the step after it. */

__global__ void __launch_bounds__(64) k_window_begin(GmDev d, uint32_t k, double xcells, uint32_t top_pos) {
    GmStats *st = d.st;
    if (top_pos < d.ndefg) {
        const uint32_t n = exact_count(d, d.rorder[top_pos]);
        if (threadIdx.x == 0) d.win->left[0] = n;
    }
    if (threadIdx.x != 0) return;
    d.win->top_hit = 0;
    st->ticket = 0;
    st->kcur = k;
    st->halt = 0;
    st->nexec = 0;
    st->ndeferred = 0;
    st->npend = 0;
    st->npend0 = 0;
    st->pone = 0;
    st->cwrap = 0;
    st->novf = 0;
    st->nplaced = 0;
    st->arr_pkey = 0ull;
    st->xcells = xcells;
}

hipError_t gm_launch_window_begin(const GmDev &d, uint32_t k, double xcells, uint32_t top_pos, hipStream_t s) {
    k_window_begin<<<1, 64, 0, s>>>(d, k, xcells, top_pos);
    return hipGetLastError();
}


/* DEFERRED cells: anchored at the step after their infection with their carry;
 * every step since then added the increment of the window's scalars, so the
 * value before step a.k is replayed from the anchor, then predicted.  The cells
 * come from the deferred list, or from a scan of every occupied slot when the
 * list overflowed. */
static __device__ __forceinline__ void predict_deferred(const GmDev &d, const GmSweepArgs &A, uint32_t i0, uint32_t stride) {
    const uint32_t nd = d.st->ndeferred;
    const bool listed = nd <= d.dlistCap;
    const uint32_t nI = d.st->nI, n = listed ? nd : nI + d.st->nB;
    for (uint32_t i = i0; i < n; i += stride) {
        const uint32_t s = listed ? d.dlist[i] : occ_slot(d, nI, i);
        if (d.cstep[s] != GM_CS_DEFERRED) continue;
        GmRec *r = d.rec + s;
        const RecA a = rec_a(r);
        const RecC c = rec_c(r);
        const double P = resolved(d, c.P);
        if (is_pending(P)) {
            atomicOr(&d.st->err, GM_ERRF_MISSED);
            continue;
        }
        r->P = P;
        double inc, f = a.frac0;
        if (cell_increment(A.sp, P, d.rho[c.defg], a.inf, inc)) f = gm_radd_n(f, inc, A.k - a.s0);
        predict_slot(d, A, s, f, A.k, P, c.defg, a.inf);
    }
}

__global__ void __launch_bounds__(GM_BLOCK) k_predict_deferred(GmDev d, GmSweepArgs A) {
    predict_deferred(d, A, blockIdx.x * GM_BLOCK + threadIdx.x, gridDim.x * GM_BLOCK);
}

/* A window's new weights into the cache and the cells that wait for them predicted, by
 * one block: few of both is the ordinary case, and two launches with a gap took 8 us
 * of it, in three steps of four on the rolled sheet. */
__global__ void __launch_bounds__(1024) k_resolve_predict(GmDev d, GmSweepArgs A, const double *vals, uint32_t npend) {
    for (uint32_t i = threadIdx.x; i < npend; i += 1024u) d.hvals[d.pend_slot[i]] = vals[i];
    __syncthreads();
    predict_deferred(d, A, threadIdx.x, 1024u);
}

hipError_t gm_launch_resolve_predict(const GmDev &d, const GmSweepArgs &a, const double *vals, uint32_t npend, hipStream_t s) {
    k_resolve_predict<<<1, 1024, 0, s>>>(d, a, vals, npend);
    return hipGetLastError();
}

hipError_t gm_launch_predict_deferred(const GmDev &d, const GmSweepArgs &a, uint32_t ndeferred, hipStream_t s) {
    if (a.nI + a.nB == 0) return hipSuccess;
    const uint32_t n = ndeferred <= d.dlistCap ? ndeferred : a.nI + a.nB;
    k_predict_deferred<<<grid_for(n, GM_BLOCK), GM_BLOCK, 0, s>>>(d, a);
    return hipGetLastError();
}

/* Cells whose weight lookup spilled (the cache had no room near the key's home):
 * with the cache grown, each looks its (nucleus, deformed grain) pair up again
 * from its record, which inserts a pending entry the host resolves before the
 * cell is predicted.  The cells come from the deferred list, or from a scan of
 * every occupied slot when the list overflowed. */
__global__ void k_spill_begin(GmDev d) {
    d.st->npend = 0;
    d.st->npend0 = 0;
    d.st->novf = 0;
}

__global__ void __launch_bounds__(GM_BLOCK) k_reinsert_spilled(GmDev d, GmPParams pp, uint32_t ndeferred, uint32_t nI,
                                                              uint32_t nB) {
    const bool listed = ndeferred <= d.dlistCap;
    const uint32_t n = listed ? ndeferred : nI + nB;
    for (uint32_t i = blockIdx.x * GM_BLOCK + threadIdx.x; i < n; i += gridDim.x * GM_BLOCK) {
        const uint32_t s = listed ? d.dlist[i] : occ_slot(d, nI, i);
        if (d.cstep[s] != GM_CS_DEFERRED) continue;
        GmRec *r = d.rec + s;
        if (!is_spilled(r->P)) continue;
        bool one = false;
        r->P = pair_weight(d, pp, r->rxg, r->defg, one);
    }
}

hipError_t gm_launch_reinsert_spilled(const GmDev &d, const GmPParams &pp, uint32_t ndeferred, uint32_t nI, uint32_t nB,
                                      hipStream_t s) {
    k_spill_begin<<<1, 1, 0, s>>>(d);
    const uint32_t n = ndeferred <= d.dlistCap ? ndeferred : nI + nB;
    if (n) k_reinsert_spilled<<<grid_for(n, GM_BLOCK), GM_BLOCK, 0, s>>>(d, pp, ndeferred, nI, nB);
    return hipGetLastError();
}
