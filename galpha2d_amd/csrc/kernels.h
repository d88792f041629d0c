// kernels.h -- launchers shared between the HIP translation units and the host orchestrator.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#define GA_INLINE_HOST_DEVICE __host__ __device__ __forceinline__

void ga_probe_begin(const char *kernel, hipStream_t st);
void ga_probe_end(const char *kernel, hipStream_t st);
// kernel launch with the optional timing probe around it
#define GA_LAUNCH(K, G, B, SH, ST, ...)                      \
    do {                                                     \
        ga_probe_begin(#K, ST);                              \
        hipLaunchKernelGGL(K, G, B, SH, ST, __VA_ARGS__);    \
        ga_probe_end(#K, ST);                                \
    } while (0)

// One point set of a batch.  Global vertex ids: the real points of all sets first (set s at
// [poff, poff + n)), then the frame vertices of all sets (set s at [fbase, fbase + nf)), so that
// inside a set the index order of the single-set layout is kept (real points before frame
// vertices, each in their own order).  Textures of all sets are concatenated in one pixel array.
struct SetDesc {
    size_t toff;         // first pixel of the set's texture
    int logT;            // texture side T = 1 << logT
    int n, poff;         // real points and the global id of the first one
    int nf, fbase;       // frame vertices and the global id of the first one
    int coff;            // first 16 x 16-pixel cell of the set (spatial numbering of the points)
    int margin;
    double shx, shy, scale, inv;   // snap grid: snapped = sh + (pixel - margin) * scale
};

// block ranges of one launch over all sets: set s owns blocks [start[s], start[s + 1])
GA_INLINE_HOST_DEVICE int set_of(const int *start, int nsets, int b)
{
    int lo = 0, hi = nsets - 1;
    while (lo < hi) {
        int mid = (lo + hi + 1) >> 1;
        if (start[mid] <= b) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

// per-launch block maps (device arrays of nsets + 1 entries each)
#define RECON_TILES 16   // 16 x 16-pixel tiles of a workgroup of the reconstruction (a 64 x 64 texture has 16)
enum { BM_COLS, BM_LABEL, BM_ROWS, BM_PIX, BM_RECON, BM_COUNT };
// rows of a block of k_pba_far_rows for a texture of side 1 << logT (0 above 4096, see pba.hip); want: rows
// for blocks enough to fill the chip
GA_INLINE_HOST_DEVICE int pba_far_rows(int logT, int want)
{
    if (logT > 12) return 0;
    const int lo = logT < 10 ? 1 << (10 - logT) : 1, hi = logT > 10 ? 1 << (14 - logT) : 16;
    return want < lo ? lo : (want > hi ? hi : want);
}
// LDS bytes of its block
inline int pba_far_lds(int T, int rows) { return 2 * T * rows * 133 / 64; }
struct BatchDev {
    const SetDesc *sets;   // [nsets]
    int nsets;
    const int *bm;         // [BM_COUNT][nsets + 1]
    int blocks[BM_COUNT];  // total blocks per map (host copy of bm[k][nsets])
    const int *vset;       // [V] set of every vertex
    int ntot, V;           // real points, all vertices
    int maxT;              // largest texture side
    int far_rows;          // rows wanted per block of k_pba_far_rows
    int far_lds;           // its largest LDS size
    size_t P;              // pixels of all textures
    GA_INLINE_HOST_DEVICE const int *bmap(int k) const { return bm + (size_t)k * (nsets + 1); }
};

struct PbaBuffers {
    int *smap;     // T*T site id per pixel (0x7fffffff = empty)
    short *g;      // T*T nearest-site row per column
    short *hmin;   // T*T/16 smallest row distance of 16 columns
    int *far;      // T*T/1024 tile parts with far pixels
    int *setfar;   // [nsets] sets with far pixels (zero on entry)
    int *vor;      // T*T nearest site id
};

// Mesh state of one point set on the device.
struct MeshDev {
    int4 *tv;            // triangle vertices (x == -2: dead slot)
    int4 *tn;            // neighbour encodings (t << 2 | j), -1 hull
    int4 *remap;         // per slot: new encoding of each old edge after a modification
    int *stamp;          // per slot: id of the last operation that modified it
    unsigned long long *claim;  // per slot: vote word
    int cap;             // slot capacity
    int *ntri;           // device: slots in use
    double2 *pos;        // current vertex positions [V]
    const double2 *xy;   // true positions of the real points [n]
    int *vt;             // vertex -> an incident triangle [V]
    int *vstate;         // vertex state [V]
    int *pix;            // vertex pixel (px << 16 | py) [V]
    int n, V;            // real points of all sets, all vertices (real + frame)
    const SetDesc *sets; // per set (snap grid, frame range, texture)
    const int *vset;     // [V] set of every vertex
    int nsets;
    int *status;         // device error bits
    int *counters;       // device scratch counters [64]; [64, 128) folded statistics
    int *stats;          // striped statistics: counters + GA_STRIPE_INTS, GA_STRIPES stripes
    int *plist;          // vertices still pending after bulk shifting (counters[C_PLIST] entries)
    const int *perm;     // input index of real vertex v (real vertices are numbered in spatial order)
    int *modA, *modB;    // modified-triangle lists (capacity cap)
    int *cand;           // candidate list (capacity 3*cap)
    int *scratch;        // per-winner scratch arena
    size_t scratch_cap;
    double *dbg;         // failure dump: positions (K + up to 15 polygon vertices) and states
    // per-context work buffers (never process globals: contexts run concurrently)
    int *deg;            // [V + 1] vertex degrees of the reconstruction
    int *mark;           // [V] state of the shifting rounds (see mesh.hip)
    const int *off;      // [V + 1] corners of every vertex in the reconstruction: fan[off[v]] .. fan[off[v + 1]]
    const int2 *fan;     // (enc(triangle, corner), next vertex)
    int *lt;             // [n] located type of every missing site
    int *lmark;          // [cap] operation that last put the slot in a flip list (one entry per pass)
    // constraint edges (set of (min << 32 | max) + 1 keys, open addressing, 0 = empty); NULL when
    // the run has no constraints.  k_flip_test never flips an edge in this set.
    const unsigned long long *chash;
    int chmask;
};

// Frame removal (see mesh.hip): the boundary vertices (real vertices of frame triangles, B of them)
// and the table of the edges to fill from.  All in buffers that are free after the flips.
struct HullBox {
    double lx, ly, hx, hy;
};
struct HullDev {
    int *ftri;                  // frame triangles (counters[C_FTRI])
    int *mark;                  // [n + 1] 1 for a boundary vertex, 3 when it has an edge to another
    int *bidx;                  // [n + 1] number of boundary vertices before v (bidx[n] = B)
    int *blist;                 // [B] boundary vertices in vertex order
    double2 *bpos;              // [B] their positions
    HullBox *bbox;              // [B / 64 + 1] boxes of 64 consecutive ones
    unsigned long long *table;  // [2 H] keys of the edges (0: free entry), then what is left of them
    int2 *list;                 // first demands and the slots of their frame triangles (counters[C_HULL])
    int *pool;                  // slots of the other frame triangles (counters[C_HULL_POOL])
    int *share;                 // HULL_SHARES counters: slots taken from each share of the pool
    unsigned long long *lines;  // [HULL_LINES] hull edges found (p << 32 | q; 0: none yet)
    int *next;                  // [2 H] links of the waves' stacks
    int room;                   // most table entries
};
#define HULL_SHARES 32
#define HULL_SHARE_INTS 32      // ints between the counters
#define HULL_LINES 32

// vertex states
#define VS_IN_MESH 1       // in the mesh, position final
#define VS_PENDING 2       // in the mesh at its snapped position
#define VS_MISSING 3       // to be inserted
#define VS_DUP 4           // exact duplicate of another point, dropped
#define VS_REMOVED 5       // frame vertex removed

// counters[] slots
#define C_FLAG 0
#define C_CAND 1
#define C_MODN 2
#define C_MODN2 3
#define C_WIN 4
#define C_SCR 5
#define C_MISS 6
#define C_SHIFTING 7          // bulk shifting has not come to an end yet
#define C_EXACT_ORIENT 8
#define C_EXACT_INCIRCLE 9
#define C_FLIPS 10
#define C_INSERTED 11
#define C_DUPS 12
#define C_FRAME 13
#define C_TESTS_INCIRCLE 14
#define C_TESTS_ORIENT 15
#define C_RECON_TRIS 16
#define C_CHANGED 17          // blocks of 1,024 pixels with some that an island repair relabelled
#define C_DELETED 18
#define C_ISLAND_SITES 19
#define C_HULL_ROOM 20        // triangle slots unused before frame removal
#define C_FLIPS_TOTAL 21
#define C_XFLIP 22            // edges left to k_flip_exact
#define C_INSERT_ROUNDS 23    // rounds run by the last k_insert_tail
#define C_FLIP_LISTED 24      // triangles listed for k_flip_test (all launches)
#define C_FTRI 25             // frame triangles listed by k_hull_scan
#define C_HULL 26             // first demands of frame removal
#define C_HULL_POOL 27        // other frame triangles (free slots)
#define C_PLEFT 28            // vertices are left to delete
#define C_MLEFT 29            // vertices are left to insert
#define C_PLIST 30            // entries of the pending-vertex list (MeshDev::plist)
#define C_RECON_STATUS 31     // status word and slot count after the reconstruction
#define C_RECON_SLOTS 39
#define C_STATUS 32           // device status word (GA_ERR_* bits); MeshDev::status points here
#define C_CONS_PEND 33        // constraints still to insert (the current insertion round's walk)
#define C_CONS_MOD 34         // slots rewritten by the current insertion round
#define C_TAIL_PASSES 35      // passes run by the last single-workgroup flip tail
#define C_TAIL_DONE 36        // 1 when that tail ended with a pass without flips
#define C_TAIL_LISTED 37      // triangles listed by flip tails (also counted in C_FLIP_LISTED)
#define C_STAR 41             // 41..43: list counts of the bulk shifting passes
#define C_LONG_RUN 44         // a run of equal 32-bit canonical keys was too long to be ordered by counting
#define FLIP_SPLIT (1 << 20)  // flip lists from this length on, and those behind passes with many exact tests, leave the
                              // exact tests to a launch of their own
#define TAIL_LIST 2048        // longest flip list the single-workgroup tail takes, and of sets of up to
#define TAIL_LIST_SMALL 16384 // INSERT_TAIL_POINTS points, whose passes cost less there than their launches
// error codes written to the device status word
#define GA_ERR_EXACT_OVERFLOW 1
#define GA_ERR_WALK 2
#define GA_ERR_RECON 4
#define GA_ERR_SCRATCH 8
#define GA_ERR_CAPACITY 16
#define GA_ERR_ISLANDS 32
#define GA_ERR_PATCH 64
// constraint insertion
#define GA_ERR_CONS_POINT 128     // a point lies inside a constraint segment
#define GA_ERR_CONS_CROSS 256     // two constraints cross
#define GA_ERR_CONS_WALK 512      // the walk along a constraint left the mesh
#define GA_ERR_CONS_DUP 1024      // a constraint endpoint is a dropped duplicate point
#define GA_ERR_CONS_TRI 2048      // a retriangulated cavity produced a triangle that is not ccw
#ifndef GA_STRIPES
#define GA_STRIPES 16         // statistic stripes, GA_STRIPE_INTS ints apart (also in dev_common.h)
#define GA_STRIPE_INTS 1024
#endif
#define C_FOLD 64             // counters[C_FOLD + k] = stripe sum of statistic k after a fold
// Counters C_EXACT_*, C_INSERTED, C_DUPS, C_TESTS_INCIRCLE, C_RECON_TRIS, C_DELETED
// and C_FLIPS_TOTAL are striped statistics (MeshDev::stats); the others are single words.
#define C_DBG 48          // 48..63: first failure dump
#define C_NCOUNTERS 64

// Sorts of up to this many pairs go by merging, longer ones by radix passes (250K points, sorts of
// 0.66M and 1.05M pairs: 283 us by merging, 231 by eight passes; 65K, 139K pairs: 57 and 85).
#define SORT_MERGE_LIMIT (512 * 1024)
// pba.hip
void launch_fill_i32(int *a, int v, size_t n, hipStream_t st);
void launch_vset(const BatchDev &b, int *vset, hipStream_t st);
// perm: input index of each real point (NULL: points in input order)
void launch_splat(const double2 *xy, const BatchDev &b, const int *perm, int *smap, int *pix, const int *fpix,
                  hipStream_t st);
// spatial numbering of the real points: perm[new] = input index, xys[new] = xy[perm[new]];
// ccount (ncells + 1 ints) zero on entry
void launch_renumber(const double2 *xy, const BatchDev &b, int *cell, int *slot, int *ccount, int *first, int ncells,
                     void *scan_tmp, int *perm, double2 *xys, hipStream_t st);
void launch_pba(const PbaBuffers &p, const int *pix, const BatchDev &b, hipStream_t st);
void launch_islands(const int *vor, const int *pix, const BatchDev &b, int *bad, int *flag, hipStream_t st);
// repairs the diagram around the sites that the certificate flagged (see pba.hip)
void launch_island_repair(const PbaBuffers &p, const BatchDev &b, int *bad, const int *pix, int *removed, int first,
                          int *rlist, int *changed, int *nchanged, int *flag, hipStream_t st);

// util.hip: up to four segments of device ints copied into one contiguous device array
struct IntSegments {
    const int *src[4];
    int len[4];
    int n;
};
void launch_gather_segments(const IntSegments &g, int *dst, hipStream_t st);
// up to 16 int arrays of any size to dst + at[k] (multiples of 4; dst: pinned host memory)
struct CopyParts {
    const int *src[16];
    size_t at[16], words[16];
    int n;
};
void launch_gather_parts(const CopyParts &g, int *dst, size_t words, hipStream_t st);
// up to 16 device int arrays, each set to one value, in one launch
struct IntFills {
    int *p[16];
    size_t len[16];
    int v[16];
    int n = 0;
    void add(void *ptr, size_t ints, int value)
    {
        p[n] = (int *)ptr;
        len[n] = ints;
        v[n] = value;
        n++;
    }
};
void launch_fill_multi(const IntFills &f, hipStream_t st);

// scan.hip
size_t scan_temp_bytes(size_t n);
void launch_exclusive_scan(const int *in, int *out, size_t n, void *temp, hipStream_t st);

// mesh.hip
void launch_recon(const int *vor, const int *pix, const BatchDev &b, MeshDev &m, int *tile_cnt, int *tile_off,
                  void *scan_tmp, hipStream_t st);
// deg, fill (V + 1 ints) zero and vt -1 on entry
void launch_adjacency(MeshDev &m, int *deg, int *off, int *fill, int2 *fan, void *scan_tmp, hipStream_t st);
// states and positions of the vertices after the reconstruction, then bulk shifting: one pass over all
// triangles (reverted vertices listed in wl_out), then passes over the stars of the vertices the previous pass listed
void launch_shift_bulk(MeshDev &m, unsigned char *moved, int *mark, int *wl_out, int cnt_out_slot,
                       int cnt_next_slot, hipStream_t st);
void launch_shift_star(MeshDev &m, unsigned char *moved, int *mark, const int *wl_in, int cnt_in_slot, int *wl_out,
                       int cnt_out_slot, int cnt_next_slot, hipStream_t st);
// once counters[cnt_slot] is zero: commits, and lists the vertices still pending into m.plist (count in
// counters[C_PLIST])
void launch_shift_commit(MeshDev &m, const unsigned char *moved, int cnt_slot, hipStream_t st);
void launch_shift_greedy(MeshDev &m, int round, int *mark, int grid, hipStream_t st);
void launch_delete_round(MeshDev &m, unsigned int *mx, int round, int grid, hipStream_t st);
// small sets (see mesh.hip): everything from the bulk passes' first worklist to the deletions, and the
// insertion rounds, one workgroup each
#define SHIFT_TAIL_POINTS 8192
#define SHIFT_TAIL_PENDING 1024
#define INSERT_TAIL_POINTS 2048
void launch_shift_tail(MeshDev &m, unsigned char *moved, int *mark, int *wlA, int *wlB, int slot, unsigned int *mx,
                       int round0, int max_rounds, bool more, hipStream_t st);
void launch_insert_tail(MeshDev &m, int *mlist, int *loc, int op0, int max_rounds, hipStream_t st);
void launch_missing_init(MeshDev &m, const int *vor, int *mlist, int *loc, hipStream_t st);
void launch_insert_round(MeshDev &m, int *mlist, int *loc, int op, int grid, hipStream_t st);
void launch_relink(MeshDev &m, const int *modlist, int cnt_slot, int op, int grid, hipStream_t st);
void launch_reset_counters(int *counters, int a, int b, int d, int e, hipStream_t st);
// counters[C_FOLD + k] = sum over the stripes of statistic k, for k < 64
void launch_fold_stats(int *counters, hipStream_t st);
// counters[slot, slot + n) (n <= 256) into pinned host memory, statistics folded when fold is set
void launch_counters_to_host(int *counters, int slot, int n, int fold, int *host, hipStream_t st);
void launch_flip_all(MeshDev &m, int op, int *list, hipStream_t st);
// flip passes on short lists in one workgroup (see k_flip_tail)
void launch_flip_tail(MeshDev &m, int *lA, int sA, int *lB, int sB, int prev_op, int op0, int max_passes,
                      int limit, hipStream_t st);
void launch_flip_pass(MeshDev &m, const int *list_in, int cnt_in_slot, int *list_out, int cnt_out_slot,
                      int prev_op, int op, int grid, bool split, hipStream_t st);
// Blocks of 256 threads for a round over about `items` list entries: enough for one entry per
// thread, a multiple of 8 (one share per XCD), at most 2048 (grid-stride loops cover any rest).
// Lists that shrink from round to round then do not launch thousands of idle blocks.
inline int round_grid(long long items)
{
    long long b = (items + 255) / 256;
    b = (b + 7) & ~7LL;
    return (int)(b < 8 ? 8 : (b > 2048 ? 2048 : b));
}
// constrained DT (see mesh.hip).  Set-up: cv = constraints as vertex ids, done flags, the key set
// (chash, size chmask + 1, cleared by the caller), vt rebuilt from the live slots.
void launch_cons_setup(MeshDev &m, const int2 *cin, int nc, int *inv, int2 *cv, int *done,
                       unsigned long long *chash, int chmask, hipStream_t st);
// one insertion round: walk (counts, region sizes) -> scan -> collect + claim -> commit -> relink
void launch_cons_count(MeshDev &m, const int2 *cv, int nc, int *done, int *cnt, int *rsize, hipStream_t st);
void launch_cons_insert(MeshDev &m, const int2 *cv, int nc, int *done, const int *cnt, const int *roff,
                        int *work, int *modlist, int op, hipStream_t st);
// frame removal (see mesh.hip); mark, share and the counters C_FTRI .. C_HULL_POOL zero on entry
void launch_hull(MeshDev &m, const HullDev &h, int op, void *scan_tmp, hipStream_t st);
// canonical order: key (v0 << B) | v1 of input indices below 2^B, sorted on its low 2B bits
// (count: the live triangles are to be counted)
void launch_canon_keys(MeshDev &m, unsigned long long *keys, int *vals, int *rot, int B, bool count, hipStream_t st);
// canonical keys of 32 bits up to input indices below 2^CANON_KEY32_BITS
#define CANON_KEY32_BITS 24
void launch_canon_keys32(MeshDev &m, unsigned *keys, unsigned *v1s, int *vals, int *rot, int B, hipStream_t st);
// out: [nslots] the order when skey is given (32-bit keys); rec: 24 bytes per slot; set_first: batches only
void launch_canon_emit(MeshDev &m, const int *order, const unsigned *skey, const unsigned *v1s, int *out, const int *rot,
                       int *newid, int2 *rec, const int *dF, int *out9, int *set_first, int *rset, hipStream_t st);
int sort_pairs_u64(unsigned long long *keys_in, int *vals_in, unsigned long long *keys_out, int *vals_out,
                   int n, int begin_bit, int end_bit, void *temp, size_t *temp_bytes, hipStream_t st);
int sort_pairs_u32(unsigned int *keys_in, int *vals_in, unsigned int *keys_out, int *vals_out,
                   int n, int begin_bit, int end_bit, void *temp, size_t *temp_bytes, hipStream_t st);
