/*
 * gm_internal.h -- device layout and kernel launchers of the growth machine.
 *
 * One domain lives in HBM as:
 *   cell   (claim, grain)[N]  the cell's infection claim key, 0xFFFFFFFF until
 *                      claimed (a claimed cell is infected in the same step and never
 *                      claimed again, so claims are never reset), beside its
 *                      deformed-grain id (< ndefg), so that one scattered load gives
 *                      both.  The id is not written during the run: only deformed
 *                      cells' are read then, and a cell that transforms is appended
 *                      to the retirement log
 *   rlog   (cell, ndefg+rxg) per retired cell in retirement order, written
 *                      coalesced with the step's parent data; the exported map
 *                      is the grid with the front's cells marked INFECTED and then
 *                      the log applied
 *   dmap   1 bit per cell, set while the cell is deformed (infectable), blocked so
 *          that one 128-byte line holds a 16x8x8 brick of cells: a 3x3x3
 *          neighbourhood usually lies in one or two lines
 *   front  Border list slots [0,capB), then from baseI on the Inside list's, which
 *          starts with what the nuclei's density asks for and grows
 *          cstep uint16[slots]   completion step (mod GM_CS_MOD) or a GM_CS_*
 *                                sentinel; the only array every step reads in full
 *          rec   GmRec[slots]    64-byte record, read and written only when a cell
 *                                is infected, predicted, re-anchored or completes
 * The two lists keep SCORE's slot numbering (SCORE_Kernel.cpp:3587-3874) so that
 * slot-level state can be compared with a serial run.
 *
 * rxFrac is kept as an anchor (frac0 at the start of step s0) plus the increment
 * inc = ((v*dt)*inv_dx) that SCORE adds every step (SCORE_Kernel.cpp:4092).  While
 * the per-step scalars stay bit-identical, rxFrac after step k is frac0 plus
 * (k-s0+1) rounded additions of inc, so the step in which it first reaches 1.0
 * (cstep) is computed in advance (gm_radd.h), and the value it then holds is
 * replayed from the anchor when the cell completes.  When any scalar changes,
 * every active cell is re-anchored with the old increment and predicted again
 * with the new one.
 */
#ifndef SCORE_GM_INTERNAL_H
#define SCORE_GM_INTERNAL_H

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <mutex>

#define GM_INFECTED 4096002000u
#define GM_FREE_CLAIM 0xFFFFFFFFu
#define GM_PENDING_TAG 0x7FF8000000000000ull  /* quiet NaN; low 32 bits carry the P-cache slot */
#define GM_PENDING_MASK 0xFFF8000000000000ull

/* Completion steps are stored in 16 bits.  A step cs is kept as cs % GM_CS_MOD
 * when it lies less than the horizon ahead of the step that predicted it, else
 * the cell is FAR; every cell is predicted again at each multiple of the
 * horizon.  So at step k every live cell's stored step lies in [k, k + horizon),
 * and cs % GM_CS_MOD names it.  A cell that completed keeps its code, which from
 * the next step on names a past step and reads as INACTIVE until a
 * re-anchoring (at the latest at the next multiple of the horizon) or a
 * defragmentation writes the INACTIVE sentinel.  Codes at or above GM_CS_MOD
 * are sentinels. */
typedef uint16_t gm_cs_t;
#define GM_CS_MOD 0x8000u
#define GM_CS_HORIZON_MAX 0x4000u  /* horizon in steps, at most GM_CS_MOD / 2 */
static_assert(GM_CS_HORIZON_MAX <= GM_CS_MOD / 2, "a past code must not wrap into the horizon before it is cleared");
#define GM_CS_INACTIVE 0xFFFFu
#define GM_CS_NEVER 0xFFFEu       /* active, does not reach rxFrac >= 1 within the run */
#define GM_CS_UNKNOWN 0xFFFDu     /* placed by nucleation, increment not yet known (the first step re-anchors) */
#define GM_CS_DEFERRED 0xFFFCu    /* mobility weight still pending: predicted at the end of the window */
#define GM_CS_FAR 0xFFFBu         /* active, completes at least a horizon after its prediction */
#define GM_STEP_NONE 0xFFFFFFFFu  /* no completion step */
#define GM_STEP_MAX 0xFFFFFFF0u   /* steps of a run stay below this */
#define GM_STEP_NEXT 0xFFFFFFFEu  /* does not complete in the predicted step; the next step predicts it again */

/* error flags raised on the device */
#define GM_ERRF_BORDER_FULL 0x1u
#define GM_ERRF_INSIDE_FULL 0x2u
#define GM_ERRF_PCACHE_FULL 0x4u
#define GM_ERRF_MISSED 0x8u       /* a prediction lies in the past: internal error */
#define GM_ERRF_KEYS 0x10u        /* more completed cells in one step than infection keys hold (2^27; 2^23 with regions) */
#define GM_ERRF_RLOG_FULL 0x20u   /* more retirements than the log holds (only cells retired twice can do it) */
#define GM_ERRF_GRID 0x80u        /* the cell grid holds an id that is no deformed grain's */
#define GM_ERRF_HALO 0x40u        /* an infection into another region found no halo to park in: internal error */

/* the mobility-weight cache probes at most this many slots from a key's home;
 * a key that finds no room within them spills: its cells hold the pending
 * marker of slot GM_OVF_SLOT and the host re-inserts them into a larger table */
#define GM_PROBE_MAX 1024u
#define GM_NO_SITE 0xFFFFFFFFu    /* a nucleus left out of the site-saturated placement */

/* order-preserving unsigned key of a double (larger value, larger key; never 0
 * for a finite value), for atomicMax over weights */
static inline __host__ __device__ unsigned long long gm_pkey(double v) {
    unsigned long long b;
    __builtin_memcpy(&b, &v, sizeof(b));
    return (b >> 63) ? ~b : (b | 0x8000000000000000ull);
}
static inline __host__ __device__ double gm_pkey_value(unsigned long long k) {
    const unsigned long long b = (k >> 63) ? (k & 0x7FFFFFFFFFFFFFFFull) : ~k;
    double v;
    __builtin_memcpy(&v, &b, sizeof(v));
    return v;
}
#define GM_OVF_SLOT 0xFFFFFFFFu

#define GM_BLOCK 256
/* The sweep reads a list in groups of GM_SW_TPC 64-slot tiles per wave; the
 * Inside list is rounded up to whole groups and the Border list's tiles follow. */
#define GM_SW_TPC 8u
static inline __host__ __device__ uint32_t gm_tiles_inside(uint32_t nI) {
    return ((nI + 63u) / 64u + GM_SW_TPC - 1u) & ~(GM_SW_TPC - 1u);
}
#define GM_MAX_BLOCKS 8192        /* grid of the partitioned passes (scanned by one 1024-thread block) */
#define GM_SCAN_BLOCKS 1024       /* fixed grid of the device-wide scans (nucleation) */
#define GM_PEND_INLINE 2048       /* new P-cache keys returned with the per-step stats */
#define GM_NK 9                   /* kernels per step (SCORE_GM_K_* order) */
#define GM_WMAX 16                /* steps per launch window at most (also below imin - 1) */
/* the window sweep of one-region handles (gm_kernels.hip) */
#define GM_SW_WAVES (GM_BLOCK / 64)
#define GM_SW_CHUNK (64u * GM_SW_TPC) /* slots a wave takes at a time */
#define GM_SW_BLOCKS 2048u        /* sweep blocks up to GM_SW_MAXCPW chunks per wave */
#define GM_SW_MAXCPW 32u
#define GM_SW_PACK 31u            /* chunks whose per-lane counts fit a byte */
#define GM_SW_FOLD 256u           /* sweep blocks up to which no scan pass runs between counting and compaction; more
                                   * in a window of few steps, while a compaction block has at most ten rows of 256
                                   * counts to add up (a scan pass takes 5 us) */
#define GM_PB 2048u               /* blocks of the propose pass at most */
#define GM_DB 1024u               /* blocks of the decide and commit passes at most */
#define GM_GRID_BLOCKS 2048u      /* blocks of the pass over the cell grid at most */
#define GM_SUBS 16u               /* parts of a deformed grain's count */
#define GM_GATT 128u              /* attempts of a chunk whose targets' grains the decide pass hands on */
#define GM_GCHUNKS 32768u         /* chunks it does that for */
#define GM_RECYCLE_BLOCKS 2048u   /* blocks of the decide launch that write recycled slots */

/* One front record: SCORE's `cell` (SCORE_Kernel.h:124-137) with rxFrac held as
 * anchor + increment.  The first 32-byte sector holds
 * what a prediction or a re-anchoring rewrites, so those write one sector. */
struct __attribute__((aligned(64))) GmRec {
    double frac0;   /* rxFrac before step s0 */
    uint32_t s0;    /* anchor step */
    uint32_t inf;   /* infector code 0..26 */
    double inc;     /* per-step increment, 0.0 when SCORE does not advance the cell */
    double spare;   /* unused, written as 0.0 with inc */
    double P;       /* mobility weight, or a pending marker */
    uint32_t cell;  /* global cell id x + y*nx + z*nx*ny */
    uint32_t defg;  /* deformed grain being consumed (mydefgid) */
    uint32_t rxg;   /* growing nucleus (myrxgid) */
    uint32_t pad[3];
};
static_assert(sizeof(GmRec) == 64, "GmRec is one 64-byte record");
/* the kernels move records as four 16-byte quarters */
static_assert(__builtin_offsetof(GmRec, inc) == 16 && __builtin_offsetof(GmRec, spare) == 24 &&
                  __builtin_offsetof(GmRec, P) == 32 && __builtin_offsetof(GmRec, cell) == 40 &&
                  __builtin_offsetof(GmRec, defg) == 44 && __builtin_offsetof(GmRec, rxg) == 48,
              "GmRec quarters: (frac0, s0, inf) | (inc, spare) | (P, cell, defg) | (rxg, pad)");

/* The completed cells of the current step, in FullRX list order (Inside list
 * first): what the infection kernels need of each parent, as three planes of
 * parentCap 16-byte entries, so that a wave's loads of one plane are contiguous.
 *   GM_PAR_IDS  (slot, cell, defg, rxg)
 *   GM_PAR_FP   (fin, P) as two doubles: rxFrac after the completing addition and
 *               the mobility weight
 *   GM_PAR_XYZ  (x, y, z, Border flag or list) */
/* with one region two planes:
 *   GM_PAR1_CELL (x | y << 16, z | Border flag << 16, defg, rxg)
 *   GM_PAR1_FP   (fin, P)
 * All are written by the propose passes. */
#define GM_PAR1_CELL 0u
#define GM_PAR1_FP 1u
#define GM_PAR1_PLANES 2u
#define GM_PAR_IDS 0u
#define GM_PAR_FP 1u
#define GM_PAR_XYZ 2u
#define GM_PAR_PLANES 3u

/* what one step of a window leaves for the host's master section */
struct GmStepRow {
    uint32_t nI, nB;          /* list lengths after the step */
    uint32_t nfullI, nfullB;
    uint32_t totRecI, totRecB;
    uint32_t recLenI, recLenB;
    uint32_t winI, winB;
    uint32_t npend;           /* P-cache entries the step inserted */
    uint32_t nattempt;
    uint32_t err;
    uint32_t nplaced;         /* nuclei placed at the start of the step */
    uint32_t pone;            /* a new pair's weight was short-circuited to 1.0 in the step */
    unsigned long long pkey;  /* largest weight of the nuclei placed in the step (gm_pkey order), 0: none */
};

struct alignas(8) GmStats {
    uint32_t nI, nB;          /* nextSlotNeverActive of both lists */
    uint32_t nfullI, nfullB;  /* parents (completed cells) of the step (several regions) */
    uint32_t totRecI, totRecB;/* INACTIVE slots seen by the sweep */
    uint32_t recLenI, recLenB;/* recycled slots available (capped) */
    uint32_t winI, winB;      /* successful infections into each list */
    uint32_t npend;           /* P-cache entries inserted this step, still unresolved */
    uint32_t err;             /* GM_ERRF_* */
    uint32_t pone;            /* set when a pair weight was short-circuited to 1.0 */
    uint32_t scan_tot[4];     /* totals written by the device-wide scans */
    uint32_t nattempt;        /* attempts that found a deformed target this step */
    uint32_t cwrap;           /* the count of a grain before the one that sets rhomax went past zero */
    uint32_t ticket;          /* blocks of the commit pass that are done (one region: of the window's last one) */
    uint32_t grow;            /* one region: the Inside slots a step's commit pass asks for before it can run */
    uint32_t need_par;        /* one region: the parents of a step that has more than the planes hold */
    uint32_t top_hit;         /* the grain that sets rhomax lost its last cell, */
    uint32_t top_next;        /* and the position of its successor in rorder (ndefg: none) */
    uint32_t dfirst;          /* defragmentation: first INACTIVE slot of the list */
    uint32_t dcount;          /* defragmentation: ACTIVE slots moved; status vector: entries */
    uint32_t novf;            /* weight lookups that found the cache full (their cells wait for a larger table) */
    uint32_t ntried;          /* with several regions: the step's attempts on deformed cells, before they are decided */
    uint32_t nplaced;         /* nuclei placed at the start of the current step */
    unsigned long long arr_pkey; /* largest weight of those nuclei (gm_pkey order) */
    unsigned long long nret;  /* entries of the retirement log (cells retired so far) */
    unsigned long long pend_keys[GM_PEND_INLINE]; /* the first new P-cache keys; all are in GmDev::pend_key */
    /* launch windows: several steps run back to back; the host reads the rows at the end */
    uint32_t kcur;            /* index of the next step */
    uint32_t halt;            /* set after a step that needs the host: later steps of the window do nothing */
    uint32_t nexec;           /* steps executed in the window */
    uint32_t ndeferred;       /* cells whose prediction waits for a pending weight */
    uint32_t npend0;          /* npend before the current step */
    double xcells;            /* Xcells, advanced by the device within a window */
    GmStepRow rows[GM_WMAX];
};

/* stop conditions of a window, checked after every step */
struct GmWindow {
    double xstop;             /* Xcells at which the host must act (termination, defragmentation) */
    uint32_t top_pos;         /* position in rorder of the grain that sets rhomax (ndefg: none) */
    uint32_t pend_limit;      /* new P-cache entries that keep the cache at most half full */
    uint32_t defer;           /* pending weights may wait for the end of the window */
    uint32_t need_one;        /* a weight of 1.0 would be the largest so far (GmStepRow::pone is only kept then) */
};

/* Parents per chunk of the decide and commit passes: a wave takes one chunk at a
 * time, a lane per parent and then a lane per winner, so a chunk aims at 52
 * winners (at 64 parents for 66 winners a second round for the last few cost as
 * much as the first), by the ratio the step before had. */
static inline __host__ __device__ uint32_t gm_chunk_size(uint32_t nfull, uint32_t nwin) {
    const uint64_t c = nwin ? (uint64_t)nfull * 52u / nwin : 64u;
    return c > 64u ? 64u : c < 16u ? 16u : (uint32_t)c;
}

/* How a window's passes are cut up, fixed over the window: sweep blocks of
 * GM_SW_WAVES waves with cpw chunks each, nbI of them over the Inside list's chI
 * chunks, the rest over the Border list's chB; W steps; blocks of the propose and
 * decide passes. */
struct GmPart {
    uint32_t nbI, nb, cpw, chI, chB, W, nbp, nbd;
    uint32_t csz0;              /* the first step's chunk size */
    uint32_t fused;             /* the compaction does the first step's propose pass */
};

/* whether compaction blocks add up the sweep blocks' counts themselves */
static inline bool gm_fold(const GmPart &P) { return P.nb <= GM_SW_FOLD || (P.W + 1u) * P.nb <= GM_SW_FOLD * 10u; }

/* the front lists as a step of the window finds them */
struct GmWinStep {
    uint32_t nI, nB;            /* list lengths */
    uint32_t totRecI, totRecB;  /* INACTIVE slots */
    uint32_t recLenI, recLenB;  /* of which may be handed out */
    uint32_t csz;               /* parents per chunk of the decide and commit passes, 16 .. 64 */
};

/* what the passes of a window share, all on the device */
struct GmWin {
    uint32_t full[GM_WMAX], fullI[GM_WMAX]; /* cells completing in each step, in all and of the Inside list */
    uint32_t off[GM_WMAX + 1];  /* completed cells before each step: its list starts at pslot[off[i]] */
    uint32_t npend0;            /* new weight-cache entries before the current step */
    uint32_t left[GM_WMAX + 1]; /* cells of the grain that sets rhomax before each step (several regions: [0], moved on;
                                 * a commit pass that runs again finds what it found) */
    uint32_t top_hit;           /* it lost its last cell */
    GmWinStep step[GM_WMAX + 1];
    unsigned long long nret0;   /* retirements before the window */
    double xcells0;             /* Xcells before the window */
};

/* Several memory regions (SCORE with OMP_NUM_THREADS = T > 1, ompshar_ca2regions,
 * SCORE_GridPartitioning.cpp:69-166).  Region r = iz*npy + iy owns front lists
 * 2r (Inside) and 2r+1 (Border), laid out one after another in the slot arrays.
 * One halo of a region (ompshar_initialize_halo, SCORE_Kernel.cpp:2085-2127): the
 * region it lies in, its origin and extent in cells (extent 0: a dummy). */
struct GmHalo {
    uint32_t inregion;
    uint16_t org[3], ext[3];
};
static_assert(sizeof(GmHalo) == 16, "GmHalo is 16 bytes");

struct alignas(16) GmRegion {
    GmHalo halo[27];            /* halo towards each neighbour; [0] unused */
    uint32_t lo[3], hi[3];      /* inclusive box */
    uint32_t nbor[27];          /* mynborregions ids: myself, faces, edges, corners */
};

/* halos an infection can be parked in (the other 18 are dummies or always
 * shadowed by one of these, which come first and span the whole x range) */
#define GM_NHALO 8
/* rows of the per-block counts of the infection pass with several regions:
 * winners into the own Inside / Border list, attempts, halo winners by halo */
#define GM_RW_I 0
#define GM_RW_B 1
#define GM_RW_A 2
#define GM_RW_H0 3
#define GM_RROWS (GM_RW_H0 + GM_NHALO)
#define GM_BCNT_ROWS 16

/* per-list tables with several regions: nlists entries, the prefix arrays nlists+1 */
struct GmLists {
    uint32_t *base;             /* first global slot of each list (multiples of 64) */
    uint32_t *cap;              /* slots of each list */
    uint32_t *rcap;             /* recycling-list capacity of each list (fixed, as SCORE's) */
    uint32_t *rbase;            /* start of each list's recycled slots in rbuf */
    uint32_t *n;                /* nextSlotNeverActive */
    uint32_t *nold;             /* the same before the current step's appends */
    uint32_t *rlen;             /* recycled slots that may be handed out this step */
    uint32_t *occ;              /* exclusive prefix of n: occupied slot i lies in list l iff occ[l] <= i < occ[l+1] */
    uint32_t *tile;             /* exclusive prefix of the sweep's tiles per list (whole 8-tile chunks) */
    uint32_t *tile_s;           /* the same as the current step's sweep saw it (tile moves on with the lengths) */
    uint32_t *par;              /* completed cells before each list's first, in FullRX order */
    uint32_t *rst;              /* INACTIVE slots before each list's first */
    uint32_t *rbuf;             /* recycled slots (list-relative), ascending per list */
    uint32_t *rs;               /* per region r (and r = T: totals), GM_RROWS prefix counts at its first parent */
    uint32_t *bstart;           /* first block of each region in the infection passes (nreg+1: blocks in use) */
    uint4 *breg;                /* each block of the infection passes (GM_MAX_BLOCKS): its parents [x, y) and region z */
    uint32_t *hoff;             /* per region, GM_NHALO offsets of the halo winners in its Border list */
};

struct GmDev {
    /* geometry */
    uint32_t nx, ny, nz, nxy;
    uint64_t N;
    uint32_t ndefg, nrxg;
    uint32_t capI, capB;        /* slots of the lists */
    uint32_t baseI;             /* first Inside slot (the Border list's 64-slot tiles come first) */
    uint32_t capImax;           /* what capI may grow to: every cell */
    uint32_t recCapI, recCapB;
    /* state */
    uint2 *cell;                /* (claim, deformed grain) per cell */
    uint2 *rlog;                /* retirement log, rlogCap entries */
    uint64_t rlogCap;
    uint32_t *dmap;
    uint32_t dnbx, dnby, dnbz;  /* bricks of the deformed-cell bitmap per axis */
    gm_cs_t *cstep;
    uint32_t horizon;           /* steps, in [16, GM_CS_HORIZON_MAX] */
    GmRec *rec;
    /* per-step lists */
    uint32_t *pslot;            /* completed cells (global slots), Inside then Border, ascending each; with one
                                 * region those of all steps of the window, step after step */
    uint4 *par;                 /* the same cells' parent data: GM_PAR_PLANES planes */
    uint32_t *recI, *recB;      /* recycled slots (list-relative), ascending, capped */
    uint64_t *mF, *mR;          /* per 64-slot tile: completed (several regions only) / INACTIVE masks */
    uint32_t *pmA;              /* per parent: ranks of its attempts on deformed cells (one region) */
    uint32_t *pmI, *pmB;        /* per parent: winning ranks into Inside / Border (several regions: pmI holds the
                                 * attempts until they are decided) */
    /* par, pmA, pmI and pmB hold parentCap entries (the parents of one step), and with
     * several regions pslot too; with one region it holds pslotCap (of a window) */
    uint32_t pslotCap;
    uint32_t *bcnt;             /* per-block counts and offsets, 8 x GM_MAX_BLOCKS */
    uint32_t *dlist;            /* slots of the cells left DEFERRED in a window (dlistCap entries) */
    uint32_t dlistCap;
    uint32_t tileCap, parentCap;
    /* window sweep (one region): rows of swb entries, one per sweep block */
    uint32_t swb;
    GmWin *win;
    uint32_t *wcnt, *wpre;      /* GM_WMAX+1 rows: cells completing in step i (row GM_WMAX: INACTIVE slots), and the
                                 * exclusive prefixes over the blocks */
    uint32_t *wwave;            /* GM_WMAX counts per wave of each block */
    uint32_t *rcnt, *rpre;      /* INACTIVE slots of each block and before it in its list; two rows, by the step's parity */
    uint32_t *rgone, *rmrg;     /* slots the step before handed out; steps whose completed cells are in the block's masks */
    uint32_t *acnt;             /* attempts per propose block, two rows by the step's parity */
    uint2 *btot;                /* winners into Inside, Border per decide block */
    uint32_t *btop;             /* parents per decide block in the grain that sets rhomax */
    uint32_t *ccnt;             /* the same per chunk of parents, Inside << 16 | Border */
    uint32_t *gatt;             /* grains of the first GM_GATT attempts' targets of the first gchunks chunks */
    uint32_t gchunks;           /* at most GM_GCHUNKS */
    /* grains */
    double *rho, *defq, *rxq;
    uint32_t *defcnt, *rxcnt;
    uint32_t *defsub;           /* GM_SUBS rows of ndefg, cells taken from defcnt since the last fold */
    uint32_t *rorder, *rpos;    /* the grains by descending rho, and each one's position */
    /* mobility-weight cache: open addressing on key rxg*ndefg+defg+1 */
    unsigned long long *hkeys;
    double *hvals;
    uint32_t hcap;
    uint32_t *pend_slot;
    unsigned long long *pend_key;
    /* nuclei arriving after step 0: pool ids grouped by step (arr_off[k] ..
     * arr_off[k+1] for step k, 1 <= k <= arr_last; arr_last 0: none), and every
     * nucleus' site and host-computed weight */
    uint32_t *arr_ids, *arr_off;
    uint32_t arr_last;
    uint32_t *nsite;
    double *nucP;
    /* nucleation scratch */
    uint32_t *nflag, *nI_, *nB_;
    uint32_t *scan_bsum;        /* 2*GM_SCAN_BLOCKS */
    GmStats *st;
    uint32_t *prog;             /* mapped host words: (steps the window has finished << 1) | halt, and whether the
                                 * stats of the window's end are in the host's mirror */
    /* several memory regions (nreg > 1); with one region none of this is used */
    uint32_t nreg, nlists;      /* T and 2T */
    uint32_t npy, npz, nry, nrz;/* region grid and slab thickness along y and z */
    GmRegion *reg;              /* nreg entries */
    GmLists L;
    uint32_t *pmH;              /* per parent: winning ranks into another region's halo */
    uint32_t *plist;            /* per parent: its list */
};

/* mobility-weight evaluation parameters the kernels need */
struct GmPParams {
    int model;                  /* 2 = Rollett-Holm: device short-circuits P == 1.0 */
    double omega_hi;            /* omega <= omega_hi  =>  P == 1.0 exactly (RH); < 0 disables */
    double fac;                 /* 1/sqrt(2) as computed by the host */
};

struct GmSweepParams {
    int model;
    double mRH, mLAGB, mHAGB, mGS;
    double Gbhalfsq, zener, dt, inv_dx;
};

/* The list lengths live on the device (GmStats nI and nB, GmWin with one region), so that a
 * window of steps runs without the host; nI and nB here only size the grids
 * (upper estimates for the window). */
struct GmSweepArgs {
    GmSweepParams sp;
    uint32_t k;                 /* step index: the window's first, a commit pass' own (several regions: st->kcur) */
    uint32_t reanchor;          /* scalars changed since the previous step */
    uint32_t nI, nB;            /* occupied slots, for the grid sizes */
    uint32_t stepcap;           /* last step a completion can fall in */
    uint32_t next_only;         /* every following step re-anchors: predict only whether a cell
                                 * completes in the step it is predicted for (else FAR) */
    uint32_t wend;              /* the step after the window (one region): no cell infected in it completes before */
};

/* launchers (gm_kernels.hip); all asynchronous on `s`.  With `ev` non-null,
 * ev[i] is recorded before kernel i of the step and ev[GM_NK] after the last. */
/* the start of a one-region window: re-anchoring (a.reanchor), the arrivals of
 * step a.k, and the window sweep */
hipError_t gm_launch_window(const GmDev &d, const GmPart &P, const GmSweepArgs &a, const GmWindow &wd, bool arrivals,
                            double xcells, hipStream_t s, hipEvent_t *ev);
/* d.defcnt brought up to date */
hipError_t gm_launch_fold_counts(const GmDev &d, hipStream_t s);
/* every active cell advanced to step a.k with its old increment and predicted again */
hipError_t gm_launch_reanchor(const GmDev &d, const GmSweepArgs &a, hipStream_t s);
/* the same two halves of a step with several regions (gm_regions.hip) */
hipError_t gm_launch_rg_sweep(const GmDev &d, const GmSweepArgs &a, uint32_t parents_upper, hipStream_t s,
                              hipEvent_t *ev);
hipError_t gm_launch_rg_infect(const GmDev &d, const GmPParams &pp, const GmSweepArgs &a, uint32_t parents_upper,
                               const GmWindow &w, GmStats *out, hipStream_t s, hipEvent_t *ev);
/* the end of a window with several regions whose last step was launched without `out` or not at all */
hipError_t gm_launch_rg_window_end(const GmDev &d, const GmWindow &w, GmStats *out, hipStream_t s);
/* with several regions: the lists' prefixes and summed lengths from d.L.n */
hipError_t gm_launch_rg_prefix(const GmDev &d, hipStream_t s);
/* with several regions: nuclei the host placed, records scattered to their slots */
hipError_t gm_launch_rg_place(const GmDev &d, const uint32_t *slots, const GmRec *recs, uint32_t n, hipStream_t s);
/* step j of a one-region window: infections and retirements; with `out` the window
 * ends with it (once a window): the last step's row, the stats into the host's mirror */
hipError_t gm_launch_infect(const GmDev &d, const GmPParams &pp, const GmSweepArgs &a, const GmPart &P,
                            const GmWindow &w, uint32_t j, GmStats *out, hipStream_t s, hipEvent_t *ev);
/* its last pass alone, after the Inside list has grown for it */
hipError_t gm_launch_commit(const GmDev &d, const GmPParams &pp, const GmSweepArgs &a, const GmPart &P,
                            const GmWindow &w, uint32_t j, GmStats *out, hipStream_t s, hipEvent_t *ev);
/* step j's parents taken back into the grains' counts: its decide pass has run, its commit pass will not */
hipError_t gm_launch_unretire(const GmDev &d, uint32_t j, hipStream_t s);
/* the end of a window whose last step was launched without it, after `launched` steps: the last step's row, the stats into the host's mirror */
hipError_t gm_launch_window_end(const GmDev &d, const GmPart &P, uint32_t launched, uint32_t top_pos, GmStats *out,
                                hipStream_t s);
/* start of a window with several regions: step index and Xcells; clears the window's accumulators */
hipError_t gm_launch_window_begin(const GmDev &d, uint32_t k, double xcells, uint32_t top_pos, hipStream_t s);
/* cells left DEFERRED in a window, with their weights now resolved: replayed to
 * step a.k under the window's scalars and predicted */
hipError_t gm_launch_predict_deferred(const GmDev &d, const GmSweepArgs &a, uint32_t ndeferred, hipStream_t s);
hipError_t gm_launch_nucleate(const GmDev &d, const uint32_t *site, const double *nucP, uint32_t nrxg, hipStream_t s);
hipError_t gm_launch_resolve_pending(const GmDev &d, const double *vals, uint32_t npend, hipStream_t s);
/* gm_launch_resolve_pending and gm_launch_predict_deferred in one, for GM_RP_MAX of each at most (at 512^3 8.0 us on
 * average below the line, the two kernels 3.6 and 6.4 us and a gap above it) */
#define GM_RP_MAX 2048u
hipError_t gm_launch_resolve_predict(const GmDev &d, const GmSweepArgs &a, const double *vals, uint32_t npend, hipStream_t s);
hipError_t gm_launch_stats_out(const GmDev &d, GmStats *out, hipStream_t s);
/* SCORE's view of slots [base, base+n) before step k, unpacked into per-field arrays */
struct GmFrontOut {
    uint8_t *act, *inf;
    uint32_t *cell, *defg, *rxg;
    double *frac, *P;
};
hipError_t gm_launch_materialize(const GmDev &d, uint32_t k, uint32_t base, uint32_t n, const GmFrontOut &o,
                                 hipStream_t s);
/* from the cell grid `src`: the cells' pairs, the deformed-cell bitmap, the grains' cell counts (d.defcnt, zeroed before) and
 * the check of the cell grid; raises GM_ERRF_GRID (d.st, zeroed before) */
hipError_t gm_launch_grid_init(const GmDev &d, const uint32_t *src, hipStream_t s);
/* ompshar_defragmentation on the list whose slot 0 is global slot `base`:
 * first_inactive leaves in st->dfirst the first INACTIVE slot in [lo, hi), or hi;
 * move compacts the ACTIVE slots of (first, nnever) to [first, first+count) through
 * the scratch records trec/tcs (nnever-first-1 entries), leaves count in st->dcount
 * and freezes the ACTIVE records left behind at their value before step k. */
hipError_t gm_launch_defrag_first_inactive(const GmDev &d, uint32_t base, uint32_t lo, uint32_t hi, uint32_t k,
                                           hipStream_t s);
hipError_t gm_launch_defrag_move(const GmDev &d, uint32_t base, uint32_t first, uint32_t nnever, uint32_t k,
                                 GmRec *trec, gm_cs_t *tcs, hipStream_t s);
/* ompcrit_clarify_status_infectedcells: (cell, grain shown) of every ACTIVE record,
 * Inside then Border, in slot order, before step k; the count goes to st->dcount.
 * ixyz and gid hold nI+nB entries. */
hipError_t gm_launch_status(const GmDev &d, uint32_t nI, uint32_t nB, uint32_t k, double thr, uint32_t *ixyz,
                            uint32_t *gid, hipStream_t s);
/* the cell grid as SCORE holds it into `out`: every cell held by an active front record
 * marked INFECTED, but every retired cell set to ndefg+rxg from the log */
hipError_t gm_launch_overlay_infected(const GmDev &d, uint32_t nI, uint32_t nB, uint32_t k, uint32_t *out,
                                      hipStream_t s);
/* that map in SCORE's raw file encoding, in place */
hipError_t gm_launch_raw2gid(uint32_t *m, uint64_t n, hipStream_t s);
hipError_t gm_launch_fill_u32(uint32_t *p, uint32_t v, size_t n, hipStream_t s);
hipError_t gm_launch_fill_u64(unsigned long long *p, unsigned long long v, size_t n, hipStream_t s);
hipError_t gm_launch_hash_insert(const GmDev &d, const unsigned long long *keys, const double *vals, uint32_t n,
                                 hipStream_t s);
/* after a window whose weight lookups spilled (st->novf): the DEFERRED cells
 * holding the spill marker look their pair up again in the (grown) cache,
 * inserting pending entries; clears st->npend and st->novf first */
/* The fixed device array of the entry point that allocates nothing
 * (gm_noalloc.hip): its address on `device`, which must be current, looked up
 * on the device's first use; `lock` holds the device's array for the caller
 * until it is released. */
hipError_t gm_scratch_acquire(int device, uint32_t **ptr, std::unique_lock<std::mutex> &lock);
hipError_t gm_launch_reinsert_spilled(const GmDev &d, const GmPParams &pp, uint32_t ndeferred, uint32_t nI, uint32_t nB,
                                      hipStream_t s);

#endif
