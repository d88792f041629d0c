// mesh.hip -- triangle-mesh stages of the Delaunay pipeline on gfx950.
//
// Reference stages replaced here (paths relative to the reference root):
//   reconstruction      Cuda/cudaReconstruction.cu:134-574 (row counting + CPU prefix + CPU hull
//                       fix + CPU vertex fans).  Here: one pass over 2x2 pixel blocks with a
//                       tile scan, triangles emitted counter-clockwise; the frame sites at the
//                       texture border make the mesh boundary a convex rectangle, so no hull fix.
//   adjacency           cpuVertexArray + kernelFindNextTriangles (:348-436): vertex fans built
//                       on the device as a CSR (degree count, scan, fill), then edge matching.
//   shifting            Cuda/cudaShifting.cu:117-599: bulk move of every vertex to its true
//                       position with exact orientation checks, then greedy independent rounds,
//                       then deletion (ear clipping of the star-shaped hole) of the rest.
//   missing insertion   Cuda/cudaMissing.cu:125-808: stochastic visibility walk, 1->3 / 2->4
//                       splits, one insertion per triangle per round by 64-bit vote words.
//   flipping            Cuda/cudaFlipping.cu:227-685: Lawson flips with an FP64 filter and an
//                       exact integer fallback on the device (no CPU pass), lifted-perturbation
//                       tie-break for co-circular quadruples.
//   boundary removal    Cuda/cudaBoundary.cu:106-608: the frame triangles are dropped at once and
//                       what they covered is filled by parallel gift wrapping.
// Links after a modification are repaired by one generic pass: a modified triangle keeps the
// old external link of each outer edge (stored as -(e+2)); if that neighbour was modified in
// the same operation the new location is read from its remap[] entry, otherwise the link is
// kept and the neighbour's back-link is written.
#include "dev_common.h"
#include "kernels.h"
#include <algorithm>

// Workgroups go to the 8 XCDs round-robin by blockIdx.x, and each XCD has its own L2.  Grid-
// stride loops give XCD k the k-th eighth of the range, and its blocks stride through that:
// neighbouring indices (triangle slots and vertices are numbered in spatial order) then share
// one L2 instead of being spread over all eight, and every XCD has the same share whatever the
// range and the grid are.  (With the k-th eighth of the blocks of every sweep instead, a list
// shorter than the grid ran on the first XCDs alone: at 65K points k_fanfill took 36 us against
// 19, a pass of k_flip_commit up to 18 against 10.)
struct XcdRange {
    int begin, end, step;
};
// of a block that takes `unit` indices per step, from its index `at` on
GA_INLINE XcdRange xcd_range(int n, int unit, int at)
{
    const int g = (int)gridDim.x, b = (int)blockIdx.x;
    if (g & 7) return {b * unit + at, n, g * unit};
    const int share = (n + 8 * unit - 1) / (8 * unit) * unit, first = (b & 7) * share;
    return {first + (b >> 3) * unit + at, first + share < n ? first + share : n, (g >> 3) * unit};
}
#define XCD_STRIDE(i, n, unit) for (auto [i, i##_end, i##_step] = xcd_range(n, unit, 0); i < i##_end; i += i##_step)
#define GRID_STRIDE(i, n) \
    for (auto [i, i##_end, i##_step] = xcd_range(n, (int)blockDim.x, (int)threadIdx.x); i < i##_end; i += i##_step)
#define FIXED_GRID 2048
#define TAIL_THREADS 1024    // of the single-workgroup insertion rounds

GA_INLINE int ic(const int4 &a, int i) { return i == 0 ? a.x : (i == 1 ? a.y : a.z); }
GA_INLINE void sc(int4 &a, int i, int v)
{
    if (i == 0) a.x = v;
    else if (i == 1) a.y = v;
    else a.z = v;
}
GA_INLINE int slot_of(const int4 &t, int v) { return t.x == v ? 0 : (t.y == v ? 1 : 2); }
GA_INLINE int mark_old(int e) { return e < 0 ? -1 : -(e + 2); }

GA_INLINE double2 snapped(const MeshDev &m, int v)
{
    const SetDesc &sd = m.sets[m.vset[v]];
    int pp = m.pix[v];
    int px = pp >> 16, py = pp & 0xffff;
    return make_double2(sd.shx + (double)(px - sd.margin) * sd.scale, sd.shy + (double)(py - sd.margin) * sd.scale);
}

// a triangle of v's set that is certainly alive while frame vertices exist: one at the set's
// first frame vertex
GA_INLINE int set_anchor(const MeshDev &m, int v) { return m.vt[m.sets[m.vset[v]].fbase]; }

// input index of vertex v: real vertices are numbered in spatial order (perm maps them back),
// frame vertices keep their ids (above every real index)
GA_INLINE int oid(const MeshDev &m, int v) { return v < m.n ? m.perm[v] : v; }

// triangle slots in use; a reservation past the capacity sets GA_ERR_CAPACITY and leaves the
// counter above it, so loops over the slots stop at the capacity until the host sees the error
GA_INLINE int ntri_used(const MeshDev &m)
{
    int n = *m.ntri;
    return n < m.cap ? n : m.cap;
}

__device__ __noinline__ int orient_slow(double2 a, double2 b, double2 c, int *status)
{
    int ovf = 0;
    int s = orient_exact(a, b, c, &ovf);
    if (ovf) atomicOr(status, GA_ERR_EXACT_OVERFLOW);
    return s;
}

GA_INLINE int orient_dev(const MeshDev &m, double2 a, double2 b, double2 c)
{
    int s = orient_filter(a, b, c);
    if (s != 0) return s;
    stat_inc(m.stats, C_EXACT_ORIENT, true);
    return orient_slow(a, b, c, m.status);
}

__device__ __noinline__ int incircle_slow(double2 a, int ia, double2 b, int ib, double2 c, int ic_,
                                          double2 d, int id, int *status)
{
    int ovf = 0;
    int s = incircle_exact_sos(a, ia, b, ib, c, ic_, d, id, &ovf);
    if (ovf) atomicOr(status, GA_ERR_EXACT_OVERFLOW);
    return s;
}

// a, b, c, d: the positions of vertices ia, ib, ic_, id, already loaded by the caller
GA_INLINE int incircle_at(const MeshDev &m, double2 a, double2 b, double2 c, double2 d, int ia, int ib,
                          int ic_, int id)
{
    int s = incircle_filter(a, b, c, d);
    if (s != 0) return s;
    stat_inc(m.stats, C_EXACT_INCIRCLE, true);
    // the symbolic tie-break ranks vertices by input index
    return incircle_slow(a, oid(m, ia), b, oid(m, ib), c, oid(m, ic_), d, oid(m, id), m.status);
}

GA_INLINE int incircle_dev(const MeshDev &m, int ia, int ib, int ic_, int id)
{
    return incircle_at(m, m.pos[ia], m.pos[ib], m.pos[ic_], m.pos[id], ia, ib, ic_, id);
}

// ---- reconstruction --------------------------------------------------------------------
// Block corners counter-clockwise: a=(x,y) b=(x+1,y) c=(x+1,y+1) d=(x,y+1).
GA_INLINE int recon_count(int a, int b, int c, int d)
{
    if (a == c || b == d) return 0;
    int neq = (a == b) + (b == c) + (c == d) + (d == a);
    if (neq >= 2) return 0;
    return neq == 1 ? 1 : 2;
}

GA_INLINE long long iorient(int pa, int pb, int pc)
{
    long long ax = pa >> 16, ay = pa & 0xffff, bx = pb >> 16, by = pb & 0xffff, cx = pc >> 16, cy = pc & 0xffff;
    return (bx - ax) * (cy - ay) - (by - ay) * (cx - ax);
}

// bits at the even positions of v, packed (inverse of the cell numbering's bit spread)
GA_INLINE unsigned compact_bits(unsigned v)
{
    v &= 0x55555555u;
    v = (v | (v >> 1)) & 0x33333333u;
    v = (v | (v >> 2)) & 0x0f0f0f0fu;
    v = (v | (v >> 4)) & 0x00ff00ffu;
    v = (v | (v >> 8)) & 0x0000ffffu;
    return v;
}

// Tiles of 16 x 16 2x2-block origins, one per 16 x 16-pixel cell, in the Morton order of the
// cells (the order the real points are numbered in), so triangles are emitted in the spatial
// order of their vertices.  A workgroup of the BM_RECON map takes RECON_TILES tiles of one set, a wave one
// tile at a time; lane k takes the four blocks at (16 cx + k / 4, 16 cy + 4 (k % 4) ..): two 16-byte
// reads and two single ones, where a thread per block read 16 labels for the same four.  Bound by
// the labels read twice and, in the emission, by the gathers of the corners' pixels (T = 4096, 1M
// points: 23 and 55 us, 43 and 85 with a thread per block and a workgroup per tile; 1,024 sets,
// 268M pixels: 437 and 676 us, 1,673 and 2,065 with a search of the sets per tile).
struct ReconLane {
    int a[5], b[5];   // labels of column x and x + 1, rows y .. y + 4
    int c[4], sum;    // triangles of the four blocks
};
GA_INLINE ReconLane recon_lane(const int *vor, int logT, int lt, int lane)
{
    ReconLane r;
    const int T = 1 << logT;
    const int x = (int)(compact_bits((unsigned)lt >> 1) << 4) + (lane >> 2);
    const int y = (int)(compact_bits((unsigned)lt) << 4) + 4 * (lane & 3);
    r.sum = 0;
    if (x < T - 1) {
        const int *p = vor + ((size_t)x << logT) + y, *q = p + T;
        const int4 u = *(const int4 *)p, w = *(const int4 *)q;
        const int more = y + 4 < T ? 4 : 3;   // the texture's last row starts no block
        r.a[0] = u.x; r.a[1] = u.y; r.a[2] = u.z; r.a[3] = u.w; r.a[4] = p[more];
        r.b[0] = w.x; r.b[1] = w.y; r.b[2] = w.z; r.b[3] = w.w; r.b[4] = q[more];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            r.c[k] = y + k < T - 1 ? recon_count(r.a[k], r.b[k], r.b[k + 1], r.a[k + 1]) : 0;
            r.sum += r.c[k];
        }
    } else {
#pragma unroll
        for (int k = 0; k < 4; k++) r.c[k] = 0;
    }
    return r;
}

__global__ __launch_bounds__(256) void k_recon_count(const int *__restrict__ vor_all, BatchDev bd,
                                                     int *__restrict__ tile_cnt)
{
    const int *bm = bd.bmap(BM_RECON);
    const int set = set_of(bm, bd.nsets, blockIdx.x);
    const SetDesc &sd = bd.sets[set];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int t0 = RECON_TILES * (int)blockIdx.x, l0 = RECON_TILES * ((int)blockIdx.x - bm[set]);
#pragma unroll
    for (int k = w; k < RECON_TILES; k += 4) {
        int s = recon_lane(vor_all + sd.toff, sd.logT, l0 + k, lane).sum;
        for (int d = 32; d > 0; d >>= 1) s += __shfl_down(s, d, 64);
        if (lane == 0) tile_cnt[t0 + k] = s;
    }
}

// the triangles of one block from slot off on; tn is left to k_match, which writes all of it
GA_INLINE void recon_emit_block(int a, int b, int cc, int d, int c, int off, const int *__restrict__ pix,
                                int4 *__restrict__ tv, int *__restrict__ status)
{
    if (c == 1) {
        int t0, t1, t2;
        if (a == b) { t0 = a; t1 = cc; t2 = d; }
        else if (b == cc) { t0 = a; t1 = b; t2 = d; }
        else { t0 = a; t1 = b; t2 = cc; }   // c == d or d == a
        if (iorient(pix[t0], pix[t1], pix[t2]) <= 0) atomicOr(status, GA_ERR_RECON);
        tv[off] = make_int4(t0, t1, t2, 0);
        return;
    }
    int pa = pix[a], pb = pix[b], pc = pix[cc], pd = pix[d];
    if (iorient(pa, pb, pc) > 0 && iorient(pa, pc, pd) > 0) {
        tv[off] = make_int4(a, b, cc, 0);
        tv[off + 1] = make_int4(a, cc, d, 0);
    } else if (iorient(pb, pc, pd) > 0 && iorient(pb, pd, pa) > 0) {
        tv[off] = make_int4(b, cc, d, 0);
        tv[off + 1] = make_int4(b, d, a, 0);
    } else {
        atomicOr(status, GA_ERR_RECON);
        tv[off] = make_int4(a, b, cc, 0);
        tv[off + 1] = make_int4(a, cc, d, 0);
    }
}

__global__ __launch_bounds__(256) void k_recon_emit(const int *__restrict__ vor_all, const int *__restrict__ pix,
                                                    BatchDev bd, const int *__restrict__ tile_cnt,
                                                    const int *__restrict__ tile_off, int4 *__restrict__ tv,
                                                    int *__restrict__ status, int *__restrict__ ntri, int cap)
{
    const int *bm = bd.bmap(BM_RECON);
    const int set = set_of(bm, bd.nsets, blockIdx.x);
    const SetDesc &sd = bd.sets[set];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int t0 = RECON_TILES * (int)blockIdx.x, l0 = RECON_TILES * ((int)blockIdx.x - bm[set]);
    if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) {
        const int last = t0 + RECON_TILES - 1;
        *ntri = min(tile_off[last] + tile_cnt[last], cap);
    }
    for (int k = w; k < RECON_TILES; k += 4) {
        if (tile_cnt[t0 + k] == 0) continue;
        const ReconLane r = recon_lane(vor_all + sd.toff, sd.logT, l0 + k, lane);
        int inc = r.sum;
        for (int d = 1; d < 64; d <<= 1) {
            const int t = __shfl_up(inc, d, 64);
            if (lane >= d) inc += t;
        }
        int off = tile_off[t0 + k] + inc - r.sum;
        if (r.sum && off + r.sum > cap) {
            atomicOr(status, GA_ERR_CAPACITY);
            continue;
        }
#pragma unroll
        for (int j = 0; j < 4; j++) {
            if (r.c[j]) recon_emit_block(r.a[j], r.b[j], r.b[j + 1], r.a[j + 1], r.c[j], off, pix, tv, status);
            off += r.c[j];
        }
    }
}

void launch_recon(const int *vor, const int *pix, const BatchDev &b, MeshDev &m, int *tile_cnt, int *tile_off,
                  void *scan_tmp, hipStream_t st)
{
    const int blocks = b.blocks[BM_RECON];
    GA_LAUNCH(k_recon_count, dim3(blocks), dim3(256), 0, st, vor, b, tile_cnt);
    launch_exclusive_scan(tile_cnt, tile_off, RECON_TILES * blocks, scan_tmp, st);
    GA_LAUNCH(k_recon_emit, dim3(blocks), dim3(256), 0, st, vor, pix, b, (const int *)tile_cnt, (const int *)tile_off,
              m.tv, m.status, m.ntri, m.cap);
}

// ---- adjacency from scratch ----------------------------------------------------------------
// Degrees and fans with the per-vertex atomics combined in LDS first.  A block takes 1024
// consecutive triangle slots; slots and vertices are both in spatial (Morton) order, so their
// vertices fall in a short id range.  Counts for ids in [vmin, vmin + ADJ_WIN) go to an LDS
// window and reach HBM as one atomic per distinct vertex and block; other ids take the global
// atomic directly.  (Device-scope atomics are performed beyond the per-XCD L2, about 11 ns each
// on one address.)
#define ADJ_WIN 8192
#define ADJ_CHUNK 1024

// smallest live vertex id of slots [c0, c0 + ADJ_CHUNK) (block-uniform; every thread calls it)
GA_INLINE int adj_chunk_min(const int4 *__restrict__ tv, int c0, int n, int *s_red)
{
    int mn = 0x7fffffff;
    for (int j = 0; j < ADJ_CHUNK / 256; j++) {
        int t = c0 + j * 256 + (int)threadIdx.x;
        if (t >= n) break;
        int4 v = tv[t];
        if (v.x == GA_DEAD) continue;
        mn = min(mn, min(v.x, min(v.y, v.z)));
    }
    for (int d = 32; d > 0; d >>= 1) mn = min(mn, __shfl_xor(mn, d, 64));
    if ((threadIdx.x & 63) == 0) s_red[threadIdx.x >> 6] = mn;
    __syncthreads();
    mn = min(min(s_red[0], s_red[1]), min(s_red[2], s_red[3]));
    return mn;
}

__global__ __launch_bounds__(256) void k_deg(const int4 *__restrict__ tv, const int *__restrict__ ntri,
                                             int *__restrict__ deg)
{
    __shared__ int cnt[ADJ_WIN];
    __shared__ int s_red[4];
    const int n = *ntri;
    XCD_STRIDE(c0, n, ADJ_CHUNK) {
        const int base = adj_chunk_min(tv, c0, n, s_red);
        for (int i = threadIdx.x; i < ADJ_WIN; i += 256) cnt[i] = 0;
        __syncthreads();
        for (int j = 0; j < ADJ_CHUNK / 256; j++) {
            int t = c0 + j * 256 + (int)threadIdx.x;
            if (t >= n) break;
            int4 v = tv[t];
            if (v.x == GA_DEAD) continue;
            for (int i = 0; i < 3; i++) {
                int a = ic(v, i);
                unsigned r = (unsigned)(a - base);
                if (r < ADJ_WIN) atomicAdd(&cnt[r], 1);
                else atomicAdd(&deg[a], 1);
            }
        }
        __syncthreads();
        for (int i = threadIdx.x; i < ADJ_WIN; i += 256) {
            int c = cnt[i];
            if (c) atomicAdd(&deg[base + i], c);
        }
        __syncthreads();
    }
}

// fan entry of corner i of triangle t: (enc(t, i), the vertex that follows it counter-clockwise);
// a corner's place in its vertex's fan is its block's base for the vertex (one global atomic per
// distinct vertex) plus its rank among the block's corners of that vertex (an LDS atomic)
__global__ __launch_bounds__(256) void k_fanfill(const int4 *__restrict__ tv, const int *__restrict__ ntri,
                                                 const int *__restrict__ off, int *__restrict__ fill,
                                                 int2 *__restrict__ fan, int *__restrict__ vt)
{
    __shared__ int cnt[ADJ_WIN];
    __shared__ int s_red[4];
    const int n = *ntri;
    XCD_STRIDE(c0, n, ADJ_CHUNK) {
        const int base = adj_chunk_min(tv, c0, n, s_red);
        for (int i = threadIdx.x; i < ADJ_WIN; i += 256) cnt[i] = 0;
        __syncthreads();
        int lr[ADJ_CHUNK / 256][3];
#pragma unroll
        for (int j = 0; j < ADJ_CHUNK / 256; j++) {
            lr[j][0] = lr[j][1] = lr[j][2] = -1;
            int t = c0 + j * 256 + (int)threadIdx.x;
            if (t >= n) continue;
            int4 v = tv[t];
            if (v.x == GA_DEAD) continue;
#pragma unroll
            for (int i = 0; i < 3; i++) {
                int a = ic(v, i);
                unsigned r = (unsigned)(a - base);
                if (r < ADJ_WIN) {
                    lr[j][i] = atomicAdd(&cnt[r], 1);
                } else {
                    int k = atomicAdd(&fill[a], 1);
                    fan[off[a] + k] = make_int2(enc(t, i), ic(v, p1(i)));
                    if (k == 0) vt[a] = t;
                }
            }
        }
        __syncthreads();
        for (int i = threadIdx.x; i < ADJ_WIN; i += 256) {
            int c = cnt[i];
            if (c) cnt[i] = atomicAdd(&fill[base + i], c);
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < ADJ_CHUNK / 256; j++) {
            int t = c0 + j * 256 + (int)threadIdx.x;
            if (t >= n) continue;
            if (lr[j][0] < 0 && lr[j][1] < 0 && lr[j][2] < 0) continue;
            int4 v = tv[t];
#pragma unroll
            for (int i = 0; i < 3; i++) {
                if (lr[j][i] < 0) continue;
                int a = ic(v, i);
                int k = cnt[a - base] + lr[j][i];
                fan[off[a] + k] = make_int2(enc(t, i), ic(v, p1(i)));
                if (k == 0) vt[a] = t;
            }
        }
        __syncthreads();
    }
}

// Edge i of t runs a -> b (a = v[i + 1], b = v[i + 2]); its twin runs b -> a in the triangle u
// whose fan entry at b has a as its next vertex, and lies opposite the corner before b in u.
__global__ void k_match(const int4 *__restrict__ tv, const int *__restrict__ ntri, const int *__restrict__ off,
                        const int2 *__restrict__ fan, int4 *__restrict__ tn)
{
    int n = *ntri;
    GRID_STRIDE(t, n) {
        int4 v = tv[t];
        if (v.x == GA_DEAD) continue;
        int4 r = make_int4(-1, -1, -1, 0);
        for (int i = 0; i < 3; i++) {
            int a = ic(v, p1(i)), b = ic(v, m1(i));
            for (int k = off[b], k1 = off[b + 1]; k < k1; k++) {
                int2 f = fan[k];
                if (f.y == a) { sc(r, i, enc(enc_t(f.x), m1(enc_j(f.x)))); break; }
            }
        }
        tn[t] = r;
    }
}

void launch_adjacency(MeshDev &m, int *deg, int *off, int *fill, int2 *fan, void *scan_tmp, hipStream_t st)
{
    GA_LAUNCH(k_deg, dim3(FIXED_GRID), dim3(256), 0, st, m.tv, m.ntri, deg);
    launch_exclusive_scan(deg, off, m.V + 1, scan_tmp, st);
    GA_LAUNCH(k_fanfill, dim3(FIXED_GRID), dim3(256), 0, st, m.tv, m.ntri, off, fill, fan, m.vt);
    GA_LAUNCH(k_match, dim3(FIXED_GRID), dim3(256), 0, st, m.tv, m.ntri, off, fan, m.tn);
}

// ---- shifting ----------------------------------------------------------------------------------
GA_INLINE double2 cand_pos(const MeshDev &m, const unsigned char *moved, int v)
{
    if (v < m.n && moved[v]) return m.xy[v];
    return m.pos[v];
}

// Bulk shifting: every pending vertex tries its true position at once (moved = 1); a triangle
// that is not counter-clockwise with the current choice reverts its moved vertices, until no
// triangle does.  Reverting only ever clears moved[], so the first pass looks at every triangle
// and later passes only at the stars of the vertices reverted by the pass before (a worklist;
// mark[] lists each vertex once).
// The first choice, with the states and positions after the reconstruction: deg (from the
// adjacency build, still valid) says which vertices are in the mesh, and every real one of these is
// pending.  Also zeroes the revert marks, the count of k_shift_bulk's output list and that of the
// first star pass's, and keeps what the reconstruction left in the slot count and the status word.
__global__ void k_shift_init(MeshDev m, const int *__restrict__ deg, unsigned char *moved, int *mark, int cnt_out_slot,
                             int cnt_next_slot)
{
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        m.counters[cnt_out_slot] = 0;
        m.counters[cnt_next_slot] = 0;
        m.counters[C_RECON_SLOTS] = *m.ntri;
        m.counters[C_RECON_STATUS] = *m.status;
    }
    GRID_STRIDE(v, m.V) {
        mark[v] = 0;
        if (v >= m.n) {
            m.vstate[v] = VS_IN_MESH;
            m.pos[v] = snapped(m, v);
            continue;
        }
        const bool in = deg[v] > 0;
        moved[v] = in ? 1 : 0;
        m.vstate[v] = in ? VS_PENDING : VS_MISSING;
        m.pos[v] = in ? snapped(m, v) : m.xy[v];
        if (!in) m.vt[v] = -1;
    }
}

// test triangle v (vertex ids) with the current choice; revert and list its moved vertices when
// it is not counter-clockwise
GA_INLINE void shift_check(const MeshDev &m, unsigned char *moved, int *mark, int4 v, int *wl_out,
                           int cnt_out_slot)
{
    bool any = (v.x < m.n && moved[v.x]) || (v.y < m.n && moved[v.y]) || (v.z < m.n && moved[v.z]);
    unsigned got = 0;   // bit k: vertex k of the triangle reverted here and listed
    if (any) {
        double2 a = cand_pos(m, moved, v.x), b = cand_pos(m, moved, v.y), cc = cand_pos(m, moved, v.z);
        if (orient_dev(m, a, b, cc) <= 0) {
#pragma unroll
            for (int k = 0; k < 3; k++) {
                int u = ic(v, k);
                if (u < m.n && moved[u]) {
                    moved[u] = 0;
                    if (atomicExch(&mark[u], 1) == 0) got |= 1u << k;
                }
            }
        }
    }
    int q = wave_reserve_n<2>(&m.counters[cnt_out_slot], __popc(got));
#pragma unroll
    for (int k = 0; k < 3; k++)
        if ((got >> k) & 1) wl_out[q++] = ic(v, k);
}

__global__ void k_shift_bulk(MeshDev m, unsigned char *moved, int *mark, int *wl_out, int cnt_out_slot)
{
    int n = ntri_used(m);
    GRID_STRIDE(t, n) {
        int4 v = m.tv[t];
        if (v.x == GA_DEAD) continue;
        shift_check(m, moved, mark, v, wl_out, cnt_out_slot);
    }
}

// Until a vertex is deleted the links are those of the reconstruction and its fans (off, fan: the
// corners of every vertex) list the stars.  Eight lanes share a star: its triangles are
// read at once, where a walk over the links is a chain of two dependent reads per triangle.
#define FAN_LANES 8

GA_INLINE void shift_star_body(const MeshDev &m, unsigned char *moved, int *mark, const int *wl_in, int nw, int *wl_out,
                               int cnt_out_slot)
{
    for (auto [k, end, step] = xcd_range(nw, (int)blockDim.x / FAN_LANES, (int)threadIdx.x / FAN_LANES); k < end; k += step) {
        int v = wl_in[k];
        for (int f = m.off[v] + threadIdx.x % FAN_LANES, f1 = m.off[v + 1]; f < f1; f += FAN_LANES)
            shift_check(m, moved, mark, m.tv[enc_t(m.fan[f].x)], wl_out, cnt_out_slot);
    }
}

// cnt_next_slot: the output count of the next pass (neither this pass's input nor its output),
// zeroed here so that no launch is needed between passes
__global__ void k_shift_star(MeshDev m, unsigned char *moved, int *mark, const int *wl_in, int cnt_in_slot,
                             int *wl_out, int cnt_out_slot, int cnt_next_slot)
{
    if (blockIdx.x == 0 && threadIdx.x == 0) m.counters[cnt_next_slot] = 0;
    shift_star_body(m, moved, mark, wl_in, m.counters[cnt_in_slot], wl_out, cnt_out_slot);
}

void launch_shift_bulk(MeshDev &m, unsigned char *moved, int *mark, int *wl_out, int cnt_out_slot,
                       int cnt_next_slot, hipStream_t st)
{
    GA_LAUNCH(k_shift_init, dim3(FIXED_GRID), dim3(256), 0, st, m, (const int *)m.deg, moved, mark, cnt_out_slot,
              cnt_next_slot);
    GA_LAUNCH(k_shift_bulk, dim3(FIXED_GRID), dim3(256), 0, st, m, moved, mark, wl_out, cnt_out_slot);
}

void launch_shift_star(MeshDev &m, unsigned char *moved, int *mark, const int *wl_in, int cnt_in_slot, int *wl_out,
                       int cnt_out_slot, int cnt_next_slot, hipStream_t st)
{
    GA_LAUNCH(k_shift_star, dim3(FIXED_GRID), dim3(256), 0, st, m, moved, mark, wl_in, cnt_in_slot, wl_out,
              cnt_out_slot, cnt_next_slot);
}

// Commits the moves once the star passes have come to an end (cnt_slot: the output count of the last
// one) and lists the few percent of the vertices that are still pending: the greedy and
// deletion rounds only look at these; a listed vertex that has left the pending state since is skipped by
// its state.  Before the end it only says so in C_SHIFTING: the list stays empty, so the
// rounds launched behind it find nothing to do.
GA_INLINE void shift_commit_body(const MeshDev &m, const unsigned char *moved)
{
    const int bd = (int)blockDim.x;
    XCD_STRIDE(b0, m.n, 4 * bd) {
        unsigned bits = 0;
        for (int j = 0; j < 4; j++) {
            int v = b0 + j * bd + (int)threadIdx.x;
            if (v >= m.n || m.vstate[v] != VS_PENDING) continue;
            if (moved[v]) {
                m.pos[v] = m.xy[v];
                m.vstate[v] = VS_IN_MESH;
            } else bits |= 1u << j;
        }
        int k = block_reserve(&m.counters[C_PLIST], __popc(bits));
        for (int j = 0; j < 4; j++)
            if ((bits >> j) & 1) m.plist[k++] = b0 + j * bd + (int)threadIdx.x;
    }
}

__global__ __launch_bounds__(256) void k_shift_commit(MeshDev m, const unsigned char *moved, int cnt_slot)
{
    const bool open = m.counters[cnt_slot] != 0;
    if (blockIdx.x == 0 && threadIdx.x == 0) m.counters[C_SHIFTING] = open;
    if (open || *m.status) return;
    shift_commit_body(m, moved);
}

void launch_shift_commit(MeshDev &m, const unsigned char *moved, int cnt_slot, hipStream_t st)
{
    GA_LAUNCH(k_shift_commit, dim3(round_grid((m.n + 3) / 4)), dim3(256), 0, st, m, moved, cnt_slot);
}

GA_INLINE uint32_t vprio(int v, int round) { return hash32((uint32_t)v * 0x9E3779B1u ^ hash32((uint32_t)round + 0x1234567u)); }

// Greedy round: a pending vertex whose pending neighbours all have lower priority moves to
// its true position when all its star triangles stay counter-clockwise.  mark[v] is 1 for a
// pending vertex (the bulk passes reverted it), round + 2 once it has moved.  Whoever was
// pending when the round began (1 or round + 2) counts as pending all round, so of two
// neighbours only the one with the higher priority can move, whether or not the other sees it
// move: one launch decides and moves.  (With one lane per vertex walking the links, and a launch
// of its own for the moves, a round took 20 us at 1M points and
// 18 at 12,007 in clusters, now 5.5 and 3.2.)
GA_INLINE bool shift_greedy_body(const MeshDev &m, int round, int *mark, int np)
{
    bool moves = false;   // this lane moved a vertex
    const int sub = threadIdx.x % FAN_LANES, shift = __lane_id() - sub;
    for (auto [k, end, step] = xcd_range(np, (int)blockDim.x / FAN_LANES, (int)threadIdx.x / FAN_LANES); k < end; k += step) {
        int v = m.plist[k];
        if (mark[v] != 1) continue;
        uint32_t p = vprio(v, round);
        double2 q = m.xy[v];
        bool no = false;
        for (int f = m.off[v] + sub, f1 = m.off[v + 1]; f < f1 && !no; f += FAN_LANES) {
            int2 e = m.fan[f];
            int a = e.y, b = ic(m.tv[enc_t(e.x)], m1(enc_j(e.x)));
            int sa = a < m.n ? mark[a] : 0;
            if (sa == 1 || sa == round + 2) {
                uint32_t pa = vprio(a, round);
                no = pa > p || (pa == p && a > v);
            }
            if (!no) no = orient_dev(m, q, m.pos[a], m.pos[b]) <= 0;
        }
        bool any = (__ballot(no) >> shift) & ((1u << FAN_LANES) - 1u);
        if (!any && sub == 0) {
            m.pos[v] = q;
            m.vstate[v] = VS_IN_MESH;
            mark[v] = round + 2;
            moves = true;
        }
    }
    return moves;
}

__global__ __launch_bounds__(256) void k_shift_greedy(MeshDev m, int round, int *mark)
{
    shift_greedy_body(m, round, mark, m.counters[C_PLIST]);
}

void launch_shift_greedy(MeshDev &m, int round, int *mark, int grid, hipStream_t st)
{
    GA_LAUNCH(k_shift_greedy, dim3(grid), dim3(256), 0, st, m, round, mark);
}

// ---- deletion of vertices that cannot move (star-shaped hole, ear clipping) --------------------
// Priorities of one round of vertex removal: the round number (< 2^20, increasing within a run)
// in the top bits, so the per-vertex maxima left by earlier rounds always lose and mx[] is
// cleared once per run; then 12 random bits; the vertex id breaks ties.
GA_INLINE unsigned long long prio64(int v, int round)
{
    return ((unsigned long long)round << 44) | ((unsigned long long)(vprio(v, round) & 0xfffu) << 32) | (unsigned)v;
}

// distance-2 independence: every vertex records the largest priority in its closed neighbourhood
GA_INLINE void del_prio_body(const MeshDev &m, unsigned long long *mx, int round, int np)
{
    GRID_STRIDE(k, np) {
        int v = m.plist[k];
        if (m.vstate[v] != VS_PENDING) continue;
        unsigned long long p = prio64(v, round);
        atomicMax(&mx[v], p);
        int t0 = m.vt[v], t = t0, i = slot_of(m.tv[t0], v), guard = 0;
        do {
            int a = ic(m.tv[t], p1(i));
            atomicMax(&mx[a], p);
            int e = ic(m.tn[t], p1(i));
            if (e < 0) { atomicOr(m.status, GA_ERR_WALK); break; }
            t = enc_t(e);
            i = p1(enc_j(e));
            if (++guard > 100000) break;
        } while (t != t0);
    }
}

// also zeroes the scratch count and the flag of pending vertices that k_del_apply of this round sets
__global__ void k_del_prio(MeshDev m, unsigned long long *mx, int round)
{
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        m.counters[C_SCR] = 0;
        m.counters[C_PLEFT] = 0;
    }
    del_prio_body(m, mx, round, m.counters[C_PLIST]);
}

// link two (triangle, slot) sides of one edge; X < 0 means hull
// single-word stores: other threads may write other slots of the same neighbour record
GA_INLINE void set_link(const MeshDev &m, int T, int k, int v) { ((int *)(m.tn + T))[k] = v; }
GA_INLINE void bond(const MeshDev &m, int T, int k, int X)
{
    set_link(m, T, k, X);
    if (X >= 0) set_link(m, enc_t(X), enc_j(X), enc(T, k));
}

// The hole is star-shaped from K (v's position): K lies left of every polygon edge.
// An ear (A, B, C) is cut when it is counter-clockwise and K is left of or on the new
// edge A -> C; that keeps K left of or on every edge of the remaining polygon, so the
// ear holds no other polygon vertex (they are in angular order around K) and an ear
// always exists.  (K strictly inside the ear is excluded by the same test.)
template <class F>
GA_INLINE void del_failed(const MeshDev &m, int v, int msz, F poly)
{
    atomicOr(m.status, GA_ERR_PATCH);
    if (atomicCAS(&m.counters[C_DBG], 0, 1) != 0) return;
    m.counters[C_DBG + 1] = v;
    m.counters[C_DBG + 2] = msz;
    for (int k = 0; k < msz && k < 12; k++) m.counters[C_DBG + 3 + k] = poly(k);
    m.dbg[0] = m.pos[v].x; m.dbg[1] = m.pos[v].y;
    for (int k = 0; k < msz && k < 15; k++) {
        m.dbg[2 + 2 * k] = m.pos[poly(k)].x;
        m.dbg[3 + 2 * k] = m.pos[poly(k)].y;
        m.dbg[32 + k] = (double)m.vstate[poly(k)];
    }
}

// one lane, any number d of corners (the polygon in the scratch arena); returns the first slot, -1 when
// the arena is full.  Inlined: a call takes the mesh by reference, so that every lane of the caller first
// stored its copy of the launch's argument, 36 MB per launch (k_del_apply 155 us of a run of 1,048,576
// points with the call and 147 registers, 105 without and with 119; 1,024 sets 1,454 and 1,080).
GA_INLINE int del_serial(const MeshDev &m, int v, int d)
{
    // scratch: poly[d], plink[d], slots[d]
    int base = atomicAdd(&m.counters[C_SCR], 3 * d);
    if ((size_t)(base + 3 * d) > m.scratch_cap) {
        atomicOr(m.status, GA_ERR_SCRATCH);
        return -1;
    }
    int *poly = m.scratch + base, *plink = poly + d, *slots = plink + d;
    int t = m.vt[v], i = slot_of(m.tv[t], v);
    for (int k = 0; k < d; k++) {
        int4 tt = m.tv[t];
        poly[k] = ic(tt, p1(i));                 // triangle (v, l_k, l_k+1)
        plink[k] = ic(m.tn[t], i);               // outer side of edge (l_k, l_k+1)
        slots[k] = t;
        int e = ic(m.tn[t], p1(i));
        t = enc_t(e);
        i = p1(enc_j(e));
    }
    double2 K = m.pos[v];
    int msz = d, used = 0;
    while (msz > 3) {
        int pick = -1;
        for (int k = 0; k < msz && pick < 0; k++) {
            int kp = k == 0 ? msz - 1 : k - 1, kn = k == msz - 1 ? 0 : k + 1;
            double2 A = m.pos[poly[kp]], B = m.pos[poly[k]], C = m.pos[poly[kn]];
            if (orient_dev(m, A, B, C) <= 0) continue;
            if (orient_dev(m, A, C, K) < 0) continue;
            pick = k;
        }
        if (pick < 0) {
            del_failed(m, v, msz, [&](int k) { return poly[k]; });
            break;
        }
        int kp = pick == 0 ? msz - 1 : pick - 1, kn = pick == msz - 1 ? 0 : pick + 1;
        int T = slots[used++];
        int A = poly[kp], B = poly[pick], C = poly[kn];
        m.tv[T] = make_int4(A, B, C, 0);
        m.tn[T] = make_int4(-1, -1, -1, 0);
        // slot 2 (opp C) = edge (A,B) -> plink[kp]; slot 0 (opp A) = edge (B,C) -> plink[pick]
        bond(m, T, 2, plink[kp]);
        bond(m, T, 0, plink[pick]);
        m.vt[A] = T; m.vt[B] = T; m.vt[C] = T;
        // new polygon edge (A, C): its other side is slot 1 (opp B) of T
        plink[kp] = enc(T, 1);
        for (int k = pick; k < msz - 1; k++) { poly[k] = poly[k + 1]; plink[k] = plink[k + 1]; }
        msz--;
    }
    if (msz == 3) {
        if (orient_dev(m, m.pos[poly[0]], m.pos[poly[1]], m.pos[poly[2]]) <= 0) atomicOr(m.status, GA_ERR_PATCH);
        int T = slots[used++];
        m.tv[T] = make_int4(poly[0], poly[1], poly[2], 0);
        m.tn[T] = make_int4(-1, -1, -1, 0);
        bond(m, T, 2, plink[0]);   // (p0,p1)
        bond(m, T, 0, plink[1]);   // (p1,p2)
        bond(m, T, 1, plink[2]);   // (p2,p0)
        m.vt[poly[0]] = T; m.vt[poly[1]] = T; m.vt[poly[2]] = T;
    }
    for (int k = used; k < d; k++) m.tv[slots[k]] = make_int4(GA_DEAD, GA_DEAD, GA_DEAD, 0);
    return slots[0];
}

// LDS written by one lane and read by another of the same wave
GA_INLINE void wave_lds_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

#define DEL_LANES 16         // lanes of a vertex
#define DEL_MAX 64           // most corners of its polygon in LDS

// Bound by dependent reads: a block takes 64 listed vertices (ENT), keeps those that hold the maximum at
// themselves, and gives each of them to 16 lanes.  One lane walks the star and puts the polygon into
// LDS; the lanes check its corners' maxima and then test all ears at once (the one with the lowest index
// is cut, and only its two neighbours are tested again).  One lane per vertex, walking the
// star twice and testing ears one after another from memory, took 37 us per round at 1M points and
// 40, up to 106, at 12,007 in clusters (long polygons), this 17 and 10, up to 40.
template <int BD, int ENT>
GA_INLINE bool del_apply_body(const MeshDev &m, const unsigned long long *mx, int round, int np)
{
    constexpr int DEL_GROUPS = BD / DEL_LANES;
    __shared__ int s_poly[DEL_GROUPS][DEL_MAX], s_link[DEL_GROUPS][DEL_MAX], s_slot[DEL_GROUPS][DEL_MAX];
    __shared__ double2 s_pos[DEL_GROUPS][DEL_MAX];
    __shared__ unsigned char s_prv[DEL_GROUPS][DEL_MAX], s_nxt[DEL_GROUPS][DEL_MAX];
    __shared__ int s_cand[ENT], s_nc;
    const int tid = threadIdx.x, grp = tid / DEL_LANES, l = tid % DEL_LANES;
    const int shift = (tid & 63) - l;
    int *poly = s_poly[grp], *link = s_link[grp], *slot = s_slot[grp];
    double2 *pos = s_pos[grp];
    unsigned char *prv = s_prv[grp], *nxt = s_nxt[grp];
    auto group = [&](bool b) { return (unsigned)(__ballot(b) >> shift) & ((1u << DEL_LANES) - 1u); };
    bool left = false;   // a vertex stays pending
    XCD_STRIDE(b0, np, ENT) {
        if (ENT > 64) {
            if (tid == 0) s_nc = 0;
            __syncthreads();
        }
        if (tid < ENT) {
            int v = b0 + tid < np ? m.plist[b0 + tid] : -1;
            bool pend = v >= 0 && m.vstate[v] == VS_PENDING, cand = pend && mx[v] == prio64(v, round);
            unsigned long long b = __ballot(cand);
            int at = 0;
            if (ENT > 64) {
                if ((tid & 63) == 0) at = atomicAdd(&s_nc, (int)__popcll(b));
                at = __shfl(at, 0, 64);
            } else if (tid == 0) {
                s_nc = __popcll(b);
            }
            if (cand) s_cand[at + __popcll(b & ((1ull << (tid & 63)) - 1ull))] = v;
            left |= pend && !cand;
        }
        __syncthreads();
        for (int q = grp, nc = s_nc; q < nc; q += DEL_GROUPS) {
            const int v = s_cand[q];
            const unsigned long long p = prio64(v, round);
            int d = 0;
            if (l == 0) {
                int t0 = m.vt[v], t = t0, i = slot_of(m.tv[t0], v);
                do {
                    int4 tt = m.tv[t], tn = m.tn[t];
                    if (d < DEL_MAX) {
                        poly[d] = ic(tt, p1(i));   // triangle (v, l_k, l_k+1)
                        link[d] = ic(tn, i);       // outer side of edge (l_k, l_k+1)
                        slot[d] = t;
                    } else if (mx[ic(tt, p1(i))] != p) { d = 0; break; }
                    int e = ic(tn, p1(i));
                    if (e < 0) { atomicOr(m.status, GA_ERR_WALK); d = 0; break; }
                    t = enc_t(e);
                    i = p1(enc_j(e));
                    if (++d > 100000) { d = 0; break; }
                } while (t != t0);
            }
            d = __shfl(d, shift, 64);
            wave_lds_sync();
            bool ok = d > 0;
            for (int k = l; k < min(d, DEL_MAX); k += DEL_LANES) {
                ok = ok && mx[poly[k]] == p;
                pos[k] = m.pos[poly[k]];
                prv[k] = (unsigned char)(k == 0 ? d - 1 : k - 1);
                nxt[k] = (unsigned char)(k == d - 1 ? 0 : k + 1);
            }
            if (group(!ok)) { left = true; continue; }
            int anchor = -1;
            if (d > DEL_MAX) {
                if (l == 0) anchor = del_serial(m, v, d);
            } else {
                wave_lds_sync();
                const double2 K = m.pos[v];
                auto ear = [&](int k) {
                    double2 A = pos[prv[k]], B = pos[k], C = pos[nxt[k]];
                    return orient_dev(m, A, B, C) > 0 && orient_dev(m, A, C, K) >= 0;
                };
                unsigned ears = 0;   // bit j: corner l + 16 j is an ear
                if (d > 3)
                    for (int k = l, j = 0; k < d; k += DEL_LANES, j++) ears |= (unsigned)ear(k) << j;
                int msz = d, used = 0, A = 0;
                for (; msz > 3; msz--, used++) {
                    int pick = -1;
                    for (int j = 0; j < DEL_MAX / DEL_LANES && pick < 0; j++) {
                        unsigned b = group((ears >> j) & 1u);
                        if (b) pick = DEL_LANES * j + __ffs((int)b) - 1;
                    }
                    if (pick < 0) break;
                    A = prv[pick];
                    const int C = nxt[pick];
                    wave_lds_sync();
                    if (l == 0) {
                        const int T = slot[used], LA = link[A], LB = link[pick];
                        const int a = poly[A], b = poly[pick], c = poly[C];
                        m.tv[T] = make_int4(a, b, c, 0);
                        // slot 2 (opposite c) = edge (a, b), slot 0 = edge (b, c), slot 1 = the new polygon edge (a, c)
                        m.tn[T] = make_int4(-1, -1, -1, 0);
                        bond(m, T, 2, LA);
                        bond(m, T, 0, LB);
                        m.vt[a] = T; m.vt[b] = T; m.vt[c] = T;
                        link[A] = enc(T, 1);
                        nxt[A] = (unsigned char)C;
                        prv[C] = (unsigned char)A;
                    }
                    wave_lds_sync();
                    if (pick % DEL_LANES == l) ears &= ~(1u << (pick / DEL_LANES));
                    if (msz > 4)
                        for (int e = 0; e < 2; e++) {
                            const int k = e ? C : A, j = k / DEL_LANES;
                            if (k % DEL_LANES == l) ears = (ears & ~(1u << j)) | ((unsigned)ear(k) << j);
                        }
                }
                if (l == 0) {
                    if (msz > 3) {
                        // the corners that are left, from A on
                        del_failed(m, v, msz, [&](int k) {
                            int x = A;
                            while (k--) x = nxt[x];
                            return poly[x];
                        });
                    } else {
                        int x = A, y = nxt[x], z = nxt[y];
                        if (orient_dev(m, pos[x], pos[y], pos[z]) <= 0) atomicOr(m.status, GA_ERR_PATCH);
                        const int T = slot[used++];
                        m.tv[T] = make_int4(poly[x], poly[y], poly[z], 0);
                        m.tn[T] = make_int4(-1, -1, -1, 0);
                        bond(m, T, 2, link[x]);   // (x, y)
                        bond(m, T, 0, link[y]);   // (y, z)
                        bond(m, T, 1, link[z]);   // (z, x)
                        m.vt[poly[x]] = T; m.vt[poly[y]] = T; m.vt[poly[z]] = T;
                    }
                    for (int k = used; k < d; k++) m.tv[slot[k]] = make_int4(GA_DEAD, GA_DEAD, GA_DEAD, 0);
                    anchor = slot[0];
                }
                wave_lds_sync();
            }
            if (l == 0 && anchor >= 0) {
                m.vstate[v] = VS_MISSING;
                m.vt[v] = anchor;      // for the re-insertion walk
                m.pos[v] = m.xy[v];
                stat_inc(m.stats, C_DELETED, true);
            }
        }
        __syncthreads();
    }
    return __syncthreads_or(left);
}

__global__ __launch_bounds__(256) void k_del_apply(MeshDev m, const unsigned long long *mx, int round)
{
    if (del_apply_body<256, 64>(m, mx, round, m.counters[C_PLIST]) && threadIdx.x == 0) m.counters[C_PLEFT] = 1;
}

// Small sets: bulk shifting from its first worklist on, the commit, the greedy rounds and the
// deletions in one workgroup, phases separated by barriers.  A launch of a few thousand lanes costs the host
// about 5 us and the device 2.5, and there are 25 of them (1,000 points: 840 us for the call with them, 770;
// 5,003 points 762 and 699); from some ten thousand points on the rounds keep more than one CU busy.
// more: only further deletion rounds (the ones before were not enough).  With more than SHIFT_TAIL_PENDING vertices
// pending the greedy and deletion rounds are left to launches of their own (8,000 points on a spiral, 3,600 of them
// pending: shifting stage 7.4 ms in one workgroup, 2.9 so).
#define SHIFT_TAIL_THREADS 512
__global__ __launch_bounds__(SHIFT_TAIL_THREADS) void k_shift_tail(MeshDev m, unsigned char *moved, int *mark, int *wlA,
                                                                   int *wlB, int slot, unsigned long long *mx, int round0,
                                                                   int max_rounds, int more)
{
    int *lin = wlA, *lout = wlB;
    for (int s = 0; !more; s++) {   // counters[slot + s % 2]: the pass's worklist (every vertex is listed once)
        const int nw = m.counters[slot + (s & 1)];
        if (nw == 0) break;
        __syncthreads();
        if (threadIdx.x == 0) m.counters[slot + 1 - (s & 1)] = 0;
        __syncthreads();
        shift_star_body(m, moved, mark, lin, nw, lout, slot + 1 - (s & 1));
        __syncthreads();
        int *t = lin; lin = lout; lout = t;
    }
    if (threadIdx.x == 0) m.counters[C_SHIFTING] = 0;
    if (__syncthreads_or(*m.status != 0)) return;
    if (!more) shift_commit_body(m, moved);
    __syncthreads();
    const int np = m.counters[C_PLIST];
    if (np > SHIFT_TAIL_PENDING) {
        if (threadIdx.x == 0) m.counters[C_PLEFT] = 1;
        return;
    }
    bool left = np > 0;
    for (int r = 0; r < 8 && left && !more; r++)
        if (!__syncthreads_or(shift_greedy_body(m, r, mark, np))) break;
    for (int r = 0; r < max_rounds && left; r++) {
        if (threadIdx.x == 0) m.counters[C_SCR] = 0;
        del_prio_body(m, mx, round0 + r, np);
        __syncthreads();
        left = del_apply_body<SHIFT_TAIL_THREADS, SHIFT_TAIL_THREADS>(m, mx, round0 + r, np);
        __syncthreads();
    }
    if (threadIdx.x == 0) m.counters[C_PLEFT] = left;
}

void launch_shift_tail(MeshDev &m, unsigned char *moved, int *mark, int *wlA, int *wlB, int slot, unsigned int *mx,
                       int round0, int max_rounds, bool more, hipStream_t st)
{
    GA_LAUNCH(k_shift_tail, dim3(1), dim3(SHIFT_TAIL_THREADS), 0, st, m, moved, mark, wlA, wlB, slot,
              (unsigned long long *)mx, round0, max_rounds, more ? 1 : 0);
}

void launch_delete_round(MeshDev &m, unsigned int *mxraw, int round, int grid, hipStream_t st)
{
    unsigned long long *mx = (unsigned long long *)mxraw;
    GA_LAUNCH(k_del_prio, dim3(grid), dim3(256), 0, st, m, mx, round);
    GA_LAUNCH(k_del_apply, dim3(std::max(8, grid / 4 & ~7)), dim3(256), 0, st, m, (const unsigned long long *)mx, round);
}

// ---- missing-site insertion ------------------------------------------------------------------
// list position k for missing vertex v and its walk start: the anchor a deleted vertex keeps,
// else a triangle of the nearest labelled pixel
GA_INLINE void missing_anchor(const MeshDev &m, const int *__restrict__ vor, int v, int k, int *mlist, int *loc)
{
    mlist[k] = v;
    // a deleted vertex keeps an anchor triangle near its old position in vt[]
    int t = m.vt[v];
    if (t < 0 || m.tv[t].x == GA_DEAD) {
        // the nearest labelled pixel (square rings around v's pixel, radius <= 16) whose
        // site is in the mesh: its triangles are next to v, so the walk stays short
        const SetDesc &sd = m.sets[m.vset[v]];
        int T = 1 << sd.logT;
        int pp = m.pix[v];
        int px = pp >> 16, py = pp & 0xffff;
        t = -1;
        for (int r = 0; r <= 16 && t < 0; r++) {
            for (int q = 0; q < (r == 0 ? 1 : 8 * r) && t < 0; q++) {
                int dx, dy;
                if (r == 0) { dx = 0; dy = 0; }
                else {
                    int side = q / (2 * r), o = q % (2 * r) - r;
                    if (side == 0) { dx = o; dy = -r; }
                    else if (side == 1) { dx = r; dy = o; }
                    else if (side == 2) { dx = -o; dy = r; }
                    else { dx = -r; dy = -o; }
                }
                int x = px + dx, y = py + dy;
                if (x < 0 || y < 0 || x >= T || y >= T) continue;
                int s = vor[sd.toff + ((size_t)x << sd.logT) + y];
                if (s >= 0 && m.vstate[s] == VS_IN_MESH) t = m.vt[s];
            }
        }
    }
    if (t < 0) t = set_anchor(m, v);
    loc[k] = t;
}

__global__ __launch_bounds__(256) void k_missing_init(MeshDev m, const int *__restrict__ vor, int *mlist, int *loc)
{
    // launched behind rounds that may not have been enough: nothing is listed then
    if (m.counters[C_SHIFTING] || m.counters[C_PLEFT] || *m.status) return;
    // block-uniform loop: 1024 vertices per block and step, one list reservation per step
    XCD_STRIDE(b0, m.n, 1024) {
        unsigned bits = 0;
        for (int j = 0; j < 4; j++) {
            int v = b0 + j * 256 + (int)threadIdx.x;
            if (v < m.n && m.vstate[v] == VS_MISSING) bits |= 1u << j;
        }
        int k0 = block_reserve(&m.counters[C_MISS], __popc(bits));
        for (int j = 0; j < 4; j++) {
            if (!((bits >> j) & 1)) continue;
            int v = b0 + j * 256 + (int)threadIdx.x;
            missing_anchor(m, vor, v, k0 + __popc(bits & ((1u << j) - 1u)), mlist, loc);
        }
    }
}

void launch_missing_init(MeshDev &m, const int *vor, int *mlist, int *loc, hipStream_t st)
{
    GA_LAUNCH(k_missing_init, dim3(FIXED_GRID), dim3(256), 0, st, m, vor, mlist, loc);
}

// located: lt = (type << 2) | edge ; type 1 inside, 2 on edge, 3 duplicate ; -1 not located
// also zeroes the modified-slot count and the flag of missing vertices that k_insert of this round
// sets (the previous round's relink, which read the count, has finished)
GA_INLINE void locate_body(const MeshDev &m, const int *mlist, int *loc, int *lt, int op, int nm)
{
    GRID_STRIDE(k, nm) {
        int v = mlist[k];
        lt[k] = -1;
        if (m.vstate[v] != VS_MISSING) continue;
        double2 p = m.xy[v];
        int t = loc[k];
        if (t < 0 || m.tv[t].x == GA_DEAD) t = set_anchor(m, v);
        uint32_t rng = hash32((uint32_t)v ^ ((uint32_t)op * 0x85ebca6bu));
        int located = 0, o[3];
        for (int step = 0; step < 4096; step++) {
            int4 tt = m.tv[t];
            rng = rng * 1664525u + 1013904223u;
            int r = (rng >> 16) % 3;
            int moved = 0;
            for (int e = 0; e < 3; e++) {
                int i = (r + e) % 3;
                o[i] = orient_dev(m, m.pos[ic(tt, p1(i))], m.pos[ic(tt, m1(i))], p);
                if (o[i] < 0) {
                    int nb = ic(m.tn[t], i);
                    if (nb < 0) { atomicOr(m.status, GA_ERR_WALK); moved = -1; break; }
                    t = enc_t(nb);
                    moved = 1;
                    break;
                }
            }
            if (moved == 0) { located = 1; break; }
            if (moved < 0) break;
        }
        loc[k] = t;
        if (!located) continue;
        int z = (o[0] == 0) + (o[1] == 0) + (o[2] == 0);
        int4 tt = m.tv[t];
        if (z >= 2) {
            int kk = o[0] != 0 ? 0 : (o[1] != 0 ? 1 : 2);
            int w = ic(tt, kk);
            m.vstate[v] = VS_DUP;
            m.vt[v] = -1 - w;      // duplicate of w
            stat_inc(m.stats, C_DUPS, true);
            continue;
        }
        unsigned long long key = ((unsigned long long)op << 32) | (0xffffffffu - (unsigned)oid(m, v));
        if (z == 0) {
            atomicMax(&m.claim[t], key);
            lt[k] = (1 << 2);
        } else {
            int i = o[0] == 0 ? 0 : (o[1] == 0 ? 1 : 2);
            int nb = ic(m.tn[t], i);
            if (nb < 0) { atomicOr(m.status, GA_ERR_WALK); continue; }
            atomicMax(&m.claim[t], key);
            atomicMax(&m.claim[enc_t(nb)], key);
            lt[k] = (2 << 2) | i;
        }
    }
}

__global__ void k_locate(MeshDev m, const int *mlist, int *loc, int *lt, int op)
{
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        m.counters[C_MODN] = 0;
        m.counters[C_MLEFT] = 0;
    }
    locate_body(m, mlist, loc, lt, op, m.counters[C_MISS]);
}

GA_INLINE bool insert_body(const MeshDev &m, const int *mlist, const int *loc, const int *lt, int op, int *list_out, int nm)
{
    bool left = false;   // a vertex stays missing
    GRID_STRIDE(k, nm) {
        int L = lt[k];
        int v = mlist[k];
        if (L < 0) {
            left |= m.vstate[v] == VS_MISSING;
            continue;
        }
        int t = loc[k];
        unsigned long long key = ((unsigned long long)op << 32) | (0xffffffffu - (unsigned)oid(m, v));
        int type = L >> 2, i = L & 3;
        int4 tt = m.tv[t], nt = m.tn[t];
        bool win = m.claim[t] == key;
        if (win && type == 2) win = m.claim[enc_t(ic(nt, i))] == key;
        // four list slots and two new triangle slots per winner, one atomic each per wave
        int q0 = wave_reserve_mult(&m.counters[C_MODN], win, 4);
        int q1 = q0 + 1, q2 = q0 + 2, q3 = q0 + 3;
        int s = wave_reserve_mult(m.ntri, win, 2);
        if (!win) {
            left = true;
            continue;
        }
        if (type == 1) {
            if (s + 2 > m.cap) {
                atomicOr(m.status, GA_ERR_CAPACITY);
                list_out[q0] = list_out[q1] = list_out[q2] = list_out[q3] = -1;
                continue;
            }
            int s1 = s, s2 = s + 1;
            int a = tt.x, b = tt.y, c = tt.z;
            m.tv[t] = make_int4(a, b, v, 0);
            m.tv[s1] = make_int4(b, c, v, 0);
            m.tv[s2] = make_int4(c, a, v, 0);
            m.tn[t] = make_int4(enc(s1, 1), enc(s2, 0), mark_old(nt.z), 0);
            m.tn[s1] = make_int4(enc(s2, 1), enc(t, 0), mark_old(nt.x), 0);
            m.tn[s2] = make_int4(enc(t, 1), enc(s1, 0), mark_old(nt.y), 0);
            m.remap[t] = make_int4(enc(s1, 2), enc(s2, 2), enc(t, 2), 0);
            m.stamp[t] = op; m.stamp[s1] = op; m.stamp[s2] = op;
            list_out[q0] = t; list_out[q1] = s1; list_out[q2] = s2; list_out[q3] = -1;
            m.vt[v] = t; m.vt[c] = s1;
        } else {
            int nb = ic(nt, i);
            int u = enc_t(nb), j = enc_j(nb);
            if (s + 2 > m.cap) {
                atomicOr(m.status, GA_ERR_CAPACITY);
                list_out[q0] = list_out[q1] = list_out[q2] = list_out[q3] = -1;
                continue;
            }
            int s1 = s, s2 = s + 1;
            int4 ut = m.tv[u], un = m.tn[u];
            int c = ic(tt, i), a = ic(tt, p1(i)), b = ic(tt, m1(i));
            int d = ic(ut, j);
            int o_bc = ic(nt, p1(i)), o_ca = ic(nt, m1(i));
            int o_ad = ic(un, p1(j)), o_db = ic(un, m1(j));
            m.tv[t] = make_int4(c, a, v, 0);
            m.tv[s1] = make_int4(c, v, b, 0);
            m.tv[u] = make_int4(d, b, v, 0);
            m.tv[s2] = make_int4(d, v, a, 0);
            m.tn[t] = make_int4(enc(s2, 0), enc(s1, 2), mark_old(o_ca), 0);
            m.tn[s1] = make_int4(enc(u, 0), mark_old(o_bc), enc(t, 1), 0);
            m.tn[u] = make_int4(enc(s1, 0), enc(s2, 2), mark_old(o_db), 0);
            m.tn[s2] = make_int4(enc(t, 0), mark_old(o_ad), enc(u, 1), 0);
            int4 rt = make_int4(0, 0, 0, 0), ru = make_int4(0, 0, 0, 0);
            sc(rt, i, -1); sc(rt, p1(i), enc(s1, 1)); sc(rt, m1(i), enc(t, 2));
            sc(ru, j, -1); sc(ru, p1(j), enc(s2, 1)); sc(ru, m1(j), enc(u, 2));
            m.remap[t] = rt; m.remap[u] = ru;
            m.stamp[t] = op; m.stamp[u] = op; m.stamp[s1] = op; m.stamp[s2] = op;
            list_out[q0] = t; list_out[q1] = s1; list_out[q2] = u; list_out[q3] = s2;
            m.vt[v] = t; m.vt[a] = t; m.vt[c] = t; m.vt[b] = u; m.vt[d] = u;
        }
        m.vstate[v] = VS_IN_MESH;
        m.pos[v] = m.xy[v];
        stat_inc(m.stats, C_INSERTED, true);
    }
    return __syncthreads_or(left);
}

__global__ void k_insert(MeshDev m, const int *mlist, const int *loc, const int *lt, int op, int *list_out)
{
    // (one store per block: a million to the one word took 0.4 ms)
    if (insert_body(m, mlist, loc, lt, op, list_out, m.counters[C_MISS]) && threadIdx.x == 0) m.counters[C_MLEFT] = 1;
}

void launch_insert_round(MeshDev &m, int *mlist, int *loc, int op, int grid, hipStream_t st)
{
    GA_LAUNCH(k_locate, dim3(grid), dim3(256), 0, st, m, (const int *)mlist, loc, m.lt, op);
    GA_LAUNCH(k_insert, dim3(grid), dim3(256), 0, st, m, (const int *)mlist, (const int *)loc,
                       (const int *)m.lt, op, m.modA);
}

// ---- generic link repair -------------------------------------------------------------------
GA_INLINE void relink_body(const MeshDev &m, const int *list, int n, int op)
{
    GRID_STRIDE(q, n) {
        int t = list[q];
        if (t < 0) continue;
        int4 r = m.tn[t];
        bool ch = false;
        for (int k = 0; k < 3; k++) {
            int e = ic(r, k);
            if (e > -2) continue;
            int old = -e - 2;
            int B = enc_t(old), jb = enc_j(old);
            if (m.stamp[B] == op) {
                sc(r, k, ic(m.remap[B], jb));
            } else {
                sc(r, k, old);
                set_link(m, B, jb, enc(t, k));
            }
            ch = true;
        }
        if (ch) m.tn[t] = r;
    }
}

__global__ void k_relink(MeshDev m, const int *list, int cnt_slot, int op, int zero_slot)
{
    int n = m.counters[cnt_slot];
    if (zero_slot >= 0 && blockIdx.x == 0 && threadIdx.x == 0) m.counters[zero_slot] = 0;
    relink_body(m, list, n, op);
}

void launch_relink(MeshDev &m, const int *modlist, int cnt_slot, int op, int grid, hipStream_t st)
{
    GA_LAUNCH(k_relink, dim3(grid), dim3(256), 0, st, m, modlist, cnt_slot, op, -1);
}

// Small sets: the insertion rounds in one workgroup until nothing is missing or max_rounds run out
__global__ __launch_bounds__(TAIL_THREADS) void k_insert_tail(MeshDev m, int *mlist, int *loc, int op0, int max_rounds)
{
    const int nm = m.counters[C_MISS];
    bool left = nm > 0;
    int r = 0;
    for (; r < max_rounds && left; r++) {
        if (threadIdx.x == 0) m.counters[C_MODN] = 0;
        locate_body(m, mlist, loc, m.lt, op0 + r, nm);
        __syncthreads();
        left = insert_body(m, mlist, loc, m.lt, op0 + r, m.modA, nm);
        relink_body(m, m.modA, m.counters[C_MODN], op0 + r);
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        m.counters[C_MLEFT] = left;
        m.counters[C_INSERT_ROUNDS] = r;
    }
}

void launch_insert_tail(MeshDev &m, int *mlist, int *loc, int op0, int max_rounds, hipStream_t st)
{
    GA_LAUNCH(k_insert_tail, dim3(1), dim3(TAIL_THREADS), 0, st, m, mlist, loc, op0, max_rounds);
}

// ---- constraint edge set ----------------------------------------------------------------------
// key of the undirected edge {a, b}; never 0 (the empty mark)
GA_INLINE unsigned long long cons_key(int a, int b)
{
    unsigned lo = (unsigned)min(a, b), hi = (unsigned)max(a, b);
    return (((unsigned long long)lo << 32) | hi) + 1ull;
}

GA_INLINE unsigned long long cons_mix(unsigned long long k)
{
    k ^= k >> 33;
    k *= 0xff51afd7ed558ccdull;
    return k ^ (k >> 33);
}

// true when {a, b} is a constraint; the table is at least twice the number of constraints, so
// every probe sequence reaches an empty slot
GA_INLINE bool cons_has(const MeshDev &m, int a, int b)
{
    unsigned long long k = cons_key(a, b);
    for (unsigned long long h = cons_mix(k);; h++) {
        unsigned long long s = m.chash[h & (unsigned long long)m.chmask];
        if (s == k) return true;
        if (s == 0) return false;
    }
}

// ---- flipping ---------------------------------------------------------------------------------
// every slot in use (dead ones are skipped by the test); no atomics: the list is the identity.
// Launched behind rounds that may not have been enough: the list is empty then.
__global__ void k_flip_all(MeshDev m, int op, int *list, int cnt_slot)
{
    const bool early = m.counters[C_SHIFTING] || m.counters[C_PLEFT] || m.counters[C_MLEFT] || *m.status;
    int n = early ? 0 : ntri_used(m);
    GRID_STRIDE(t, n) {
        m.stamp[t] = op;
        list[t] = t;
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        m.counters[cnt_slot] = n;
        m.counters[C_CAND] = 0;
    }
}

void launch_flip_all(MeshDev &m, int op, int *list, hipStream_t st)
{
    GA_LAUNCH(k_flip_all, dim3(FIXED_GRID), dim3(256), 0, st, m, op, list, C_MODN);
}

// Candidates are the listed triangles' edges that fail the incircle test (each edge once: the
// lower slot of a pair that were both modified in the previous pass skips it).  Block-uniform
// loop over 256 * per list entries per block and step with one reservation of candidate slots
// per step: per = 4 for lists longer than four times the grid (fewer reservations), else 1 (more
// waves in flight for the latency-bound gathers).
// block-uniform: every thread of the block runs the same iterations (block_reserve inside)
// SPLIT: edges that the filter leaves open are listed in m.scratch (an edge is tested from at most
// two sides: 6 V entries; counters[C_XFLIP]) for k_flip_exact.  The exact test takes registers and
// scratch memory that leave three waves per SIMD to the whole kernel, and on a lattice a few lanes
// of every wave take it (first pass at 1M uniform points: 117 us, 80 split; the passes over a
// lattice and clusters of 2M points together 2,600 us, 1,470 split).  Lists of less than FLIP_SPLIT
// triangles keep it inside unless the passes before took many exact tests: the launch more costs
// what it gives there (250K points in clusters: 3.35 ms, all passes split 3.44).
template <bool SPLIT>
GA_INLINE void flip_test_body(const MeshDev &m, const int *list, int n, int prev_op, int op)
{
    int tests = 0;
    const int bd = (int)blockDim.x;
    int per = n > 4 * (int)(gridDim.x * bd) ? 4 : 1;
    XCD_STRIDE(b0, n, bd * per) {
        unsigned bits = 0;   // bit 3j + i: edge i of the j-th triangle of this thread wants a flip
        unsigned open = 0;   // the same: the filter leaves it open
        int tj[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            tj[j] = -1;
            if (j >= per) continue;
            int q = b0 + j * bd + (int)threadIdx.x;
            int t = q < n ? list[q] : -1;
            tj[j] = t;
            if (t < 0) continue;
            int4 tt = m.tv[t];
            if (tt.x == GA_DEAD) continue;
            int4 nn = m.tn[t];
            // The edges to test first, then every gather they need before any predicate: the
            // corner positions once, the three opposite vertices, then their positions, so the
            // three dependent chains are in flight together instead of one after another behind
            // the claim atomics.
            int uu[3];
#pragma unroll
            for (int i = 0; i < 3; i++) {
                int e = ic(nn, i);
                uu[i] = -1;
                if (e < 0) continue;
                int u = enc_t(e);
                if (m.stamp[u] == prev_op && u < t) continue;
                if (m.chash && cons_has(m, ic(tt, p1(i)), ic(tt, m1(i)))) continue;   // constraint edge
                uu[i] = u;
            }
            if ((uu[0] & uu[1] & uu[2]) < 0) continue;   // no edge to test
            int dd[3];
#pragma unroll
            for (int i = 0; i < 3; i++) dd[i] = uu[i] >= 0 ? ic(m.tv[uu[i]], enc_j(ic(nn, i))) : 0;
            double2 pa = m.pos[tt.x], pb = m.pos[tt.y], pc = m.pos[tt.z];
            double2 pd[3];
#pragma unroll
            for (int i = 0; i < 3; i++) pd[i] = uu[i] >= 0 ? m.pos[dd[i]] : make_double2(0.0, 0.0);
#pragma unroll
            for (int i = 0; i < 3; i++) {
                if (uu[i] < 0) continue;
                tests++;
                int in;
                if (SPLIT) {
                    in = incircle_filter(pa, pb, pc, pd[i]);
                    open |= (unsigned)(in == 0) << (3 * j + i);
                } else {
                    in = incircle_at(m, pa, pb, pc, pd[i], tt.x, tt.y, tt.z, dd[i]);
                }
                if (in > 0) {
                    unsigned long long key = ((unsigned long long)op << 32) | (0xffffffffu - (unsigned)(t * 3 + i));
                    atomicMax(&m.claim[t], key);
                    atomicMax(&m.claim[uu[i]], key);
                    bits |= 1u << (3 * j + i);
                }
            }
        }
        int slot = block_reserve(&m.counters[C_CAND], __popc(bits));
#pragma unroll
        for (int j = 0; j < 4; j++)
            for (int i = 0; i < 3; i++)
                if ((bits >> (3 * j + i)) & 1) m.cand[slot++] = tj[j] * 3 + i;
        if (SPLIT && __syncthreads_or(open)) {
            slot = block_reserve(&m.counters[C_XFLIP], __popc(open));
#pragma unroll
            for (int j = 0; j < 4; j++)
                for (int i = 0; i < 3; i++)
                    if ((open >> (3 * j + i)) & 1) m.scratch[slot++] = tj[j] * 3 + i;
        }
    }
    stat_add_full(m.stats, C_TESTS_INCIRCLE, tests);
}

template <bool SPLIT>
__global__ __launch_bounds__(256) void k_flip_test(MeshDev m, const int *list, int cnt_slot, int prev_op, int op,
                                                   int cnt_out_slot)
{
    int n = m.counters[cnt_slot];
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        atomicAdd(&m.counters[C_FLIP_LISTED], n);
        // the commit of this pass counts its output list and its flips from zero
        m.counters[cnt_out_slot] = 0;
        m.counters[C_FLIPS] = 0;
    }
    flip_test_body<SPLIT>(m, list, n, prev_op, op);
}

// the edges that k_flip_test<true> left open
__global__ __launch_bounds__(256) void k_flip_exact(MeshDev m, int op)
{
    const int n = m.counters[C_XFLIP];
    GRID_STRIDE(k, n) {
        const int c = m.scratch[k], t = c / 3, i = c % 3;
        const int4 tt = m.tv[t];
        const int e = ic(m.tn[t], i), u = enc_t(e), d = ic(m.tv[u], enc_j(e));
        stat_inc(m.stats, C_EXACT_INCIRCLE, true);
        const bool in = incircle_slow(m.pos[tt.x], oid(m, tt.x), m.pos[tt.y], oid(m, tt.y), m.pos[tt.z], oid(m, tt.z),
                                      m.pos[d], oid(m, d), m.status) > 0;
        const int slot = wave_reserve(&m.counters[C_CAND], in);
        if (!in) continue;
        const unsigned long long key = ((unsigned long long)op << 32) | (0xffffffffu - (unsigned)c);
        atomicMax(&m.claim[t], key);
        atomicMax(&m.claim[u], key);
        m.cand[slot] = c;
    }
}


// Block-uniform loop (block_reserve inside): up to four candidates per thread and step, and one
// reservation of output-list slots per block and step (a reservation per wave put thousands of
// atomics on the one counter).
GA_INLINE void flip_commit_body(const MeshDev &m, int n, int op, int *list_out, int cnt_out_slot)
{
    int flips = 0;
    const int bd = (int)blockDim.x;
    const int per = n > 4 * (int)(gridDim.x * bd) ? 4 : 1;
    XCD_STRIDE(b0, n, bd * per) {
        int tq[4], uq[4];
        unsigned outs = 0;   // bit 2j: slot t of the j-th candidate joins the next list, 2j + 1: slot u
#pragma unroll
        for (int j = 0; j < 4; j++) {
            tq[j] = 0;
            uq[j] = 0;
            if (j >= per) continue;
            int q = b0 + j * bd + (int)threadIdx.x;
            if (q >= n) continue;
            int c = m.cand[q];
            int t = c / 3, i = c % 3;
            unsigned long long key = ((unsigned long long)op << 32) | (0xffffffffu - (unsigned)c);
            bool win = m.claim[t] == key;
            int4 tt = m.tv[t], nt = m.tn[t];
            int e = ic(nt, i);
            int u = enc_t(e), jj = enc_j(e);
            win = win && m.claim[u] == key;
            // Next pass's list: both triangles of a flip, and the first triangle of a losing
            // candidate (its edge may stay non-Delaunay when the candidate that beat it lost too);
            // lmark keeps every slot at most once per list, so no candidate key repeats.
            if (atomicExch(&m.lmark[t], op) != op) outs |= 1u << (2 * j);
            if (win && atomicExch(&m.lmark[u], op) != op) outs |= 2u << (2 * j);
            tq[j] = t;
            uq[j] = u;
            if (!win) continue;
            int4 ut = m.tv[u], un = m.tn[u];
            int cc = ic(tt, i), x = ic(tt, p1(i)), y = ic(tt, m1(i));
            int d = ic(ut, jj);
            int nt1 = ic(nt, p1(i)), nt2 = ic(nt, m1(i));   // (y,c) , (c,x)
            int nu1 = ic(un, p1(jj)), nu2 = ic(un, m1(jj));   // (x,d) , (d,y)
            m.tv[t] = make_int4(cc, x, d, 0);
            m.tv[u] = make_int4(d, y, cc, 0);
            m.tn[t] = make_int4(mark_old(nu1), enc(u, 1), mark_old(nt2), 0);
            m.tn[u] = make_int4(mark_old(nt1), enc(t, 1), mark_old(nu2), 0);
            int4 rt = make_int4(0, 0, 0, 0), ru = make_int4(0, 0, 0, 0);
            sc(rt, i, -1); sc(rt, p1(i), enc(u, 0)); sc(rt, m1(i), enc(t, 2));
            sc(ru, jj, -1); sc(ru, p1(jj), enc(t, 0)); sc(ru, m1(jj), enc(u, 2));
            m.remap[t] = rt; m.remap[u] = ru;
            m.stamp[t] = op; m.stamp[u] = op;
            m.vt[x] = t; m.vt[cc] = t; m.vt[y] = u; m.vt[d] = u;
            flips++;
        }
        int slot = block_reserve(&m.counters[cnt_out_slot], __popc(outs));
#pragma unroll
        for (int j = 0; j < 4; j++) {
            if ((outs >> (2 * j)) & 1) list_out[slot++] = tq[j];
            if ((outs >> (2 * j + 1)) & 1) list_out[slot++] = uq[j];
        }
    }
    // C_FLIPS only tells the host whether the pass flipped anything: a plain store
    int wf = flips;
    for (int d = 32; d > 0; d >>= 1) wf += __shfl_xor(wf, d, 64);
    if (__lane_id() == 0 && wf) m.counters[C_FLIPS] = 1;
    stat_add_full(m.stats, C_FLIPS_TOTAL, flips);
}

__global__ void k_flip_commit(MeshDev m, int op, int *list_out, int cnt_out_slot)
{
    if (blockIdx.x == 0 && threadIdx.x == 0) m.counters[C_XFLIP] = 0;
    flip_commit_body(m, m.counters[C_CAND], op, list_out, cnt_out_slot);
}

// Short lists: the remaining passes in one workgroup, phases separated by block barriers instead
// of launches, until a pass flips nothing (counters[C_TAIL_DONE] = 1) or the list outgrows
// limit or max_passes run out (the host goes on with grid passes).  Pass k uses op op0 + k;
// counters[C_TAIL_PASSES] = passes run (odd: the lists have swapped).
// 512 threads: the exact test needs 174 registers, and 1,024 leave 128 (305 spilled).  All passes of 1,000
// points 91 -> 59 us, of 12,007 in clusters 171 -> 111; with the exact tests as a step of their own 106 and
// 202 (1,024 threads), 65 and 126 (512), at 256 threads without it 69 and 122.
// Small sets (limit above TAIL_LIST) with more than three points of four inserted leave long lists to grid passes as
// well: their points lie far closer together than the pixels, their exact tests need the big integers, and these
// come one after another in every wave (2,000 points, all but two within 1e-9 of the set's size: all passes 8.2 ms, 5.7
// so).
#define FLIP_TAIL_THREADS 512
__global__ __launch_bounds__(FLIP_TAIL_THREADS) void k_flip_tail(MeshDev m, int *lA, int sA, int *lB, int sB,
                                                                 int prev_op, int op0, int max_passes, int limit)
{
    int *lin = lA, *lout = lB, sin = sA, sout = sB;
    int prev = prev_op, pass = 0, done = 0;
    if (4 * m.counters[C_MISS] > 3 * m.n) limit = min(limit, TAIL_LIST);
    for (; pass < max_passes; pass++) {
        const int n = m.counters[sin];
        if (n > limit) break;
        const int op = op0 + pass;
        __syncthreads();   // every thread has read n before the counters are reset
        if (threadIdx.x == 0) {
            atomicAdd(&m.counters[C_FLIP_LISTED], n);
            atomicAdd(&m.counters[C_TAIL_LISTED], n);
            m.counters[sout] = 0;
            m.counters[C_CAND] = 0;
            m.counters[C_FLIPS] = 0;
        }
        __syncthreads();
        flip_test_body<false>(m, lin, n, prev, op);
        __syncthreads();
        flip_commit_body(m, m.counters[C_CAND], op, lout, sout);
        __syncthreads();
        relink_body(m, lout, m.counters[sout], op);
        __syncthreads();
        const bool any = m.counters[C_FLIPS] != 0;
        prev = op;
        int *tl = lin; lin = lout; lout = tl;
        int ts = sin; sin = sout; sout = ts;
        if (!any) {
            pass++;
            done = 1;
            break;
        }
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        m.counters[C_CAND] = 0;
        m.counters[C_TAIL_PASSES] = pass;
        m.counters[C_TAIL_DONE] = done;
    }
}

void launch_flip_tail(MeshDev &m, int *lA, int sA, int *lB, int sB, int prev_op, int op0, int max_passes,
                      int limit, hipStream_t st)
{
    GA_LAUNCH(k_flip_tail, dim3(1), dim3(FLIP_TAIL_THREADS), 0, st, m, lA, sA, lB, sB, prev_op, op0, max_passes,
              limit);
}

// Three launches per pass (four with the exact tests split off) and no counter resets of their own: the test clears the output list's
// count and the flip flag, and the relink clears the candidate count for the next pass (it must
// be zero before the first pass).
void launch_flip_pass(MeshDev &m, const int *list_in, int cnt_in_slot, int *list_out, int cnt_out_slot,
                      int prev_op, int op, int grid, bool split, hipStream_t st)
{
    if (split) {
        GA_LAUNCH(k_flip_test<true>, dim3(grid), dim3(256), 0, st, m, list_in, cnt_in_slot, prev_op, op, cnt_out_slot);
        GA_LAUNCH(k_flip_exact, dim3(std::min(grid, 512)), dim3(256), 0, st, m, op);
    } else {
        GA_LAUNCH(k_flip_test<false>, dim3(grid), dim3(256), 0, st, m, list_in, cnt_in_slot, prev_op, op, cnt_out_slot);
    }
    GA_LAUNCH(k_flip_commit, dim3(grid), dim3(256), 0, st, m, op, list_out, cnt_out_slot);
    GA_LAUNCH(k_relink, dim3(grid), dim3(256), 0, st, m, (const int *)list_out, cnt_out_slot, op, C_CAND);
}

// zero up to four counter slots in one launch (negative slot: unused)
__global__ void k_reset_counters(int *c, int a, int b, int d, int e)
{
    if (threadIdx.x == 0) {
        if (a >= 0) c[a] = 0;
        if (b >= 0) c[b] = 0;
        if (d >= 0) c[d] = 0;
        if (e >= 0) c[e] = 0;
    }
}

void launch_reset_counters(int *counters, int a, int b, int d, int e, hipStream_t st)
{
    GA_LAUNCH(k_reset_counters, dim3(1), dim3(64), 0, st, counters, a, b, d, e);
}

__global__ void k_fold_stats(int *c)
{
    int k = threadIdx.x, sum = 0;
    for (int s = 0; s < GA_STRIPES; s++) sum += c[GA_STRIPE_INTS * (1 + s) + k];
    c[C_FOLD + k] = sum;
}

void launch_fold_stats(int *counters, hipStream_t st)
{
    GA_LAUNCH(k_fold_stats, dim3(1), dim3(64), 0, st, counters);
}

// counters[slot, slot + n) straight into pinned host memory (n <= 256); with fold, the slots
// C_FOLD + k hold the stripe sum of statistic k (also stored back on the device, as k_fold_stats
// does).  The host waits on the stream before it reads.
__global__ void k_counters_to_host(int *c, int slot, int n, int fold, int *host)
{
    const int i = threadIdx.x;
    if (i < n) {
        const int q = slot + i;
        int v;
        if (fold && q >= C_FOLD && q < C_FOLD + 64) {
            v = 0;
            for (int s = 0; s < GA_STRIPES; s++) v += c[GA_STRIPE_INTS * (1 + s) + (q - C_FOLD)];
            c[q] = v;
        } else {
            v = c[q];
        }
        host[i] = v;
    }
    __threadfence_system();
}

void launch_counters_to_host(int *counters, int slot, int n, int fold, int *host, hipStream_t st)
{
    GA_LAUNCH(k_counters_to_host, dim3(1), dim3(256), 0, st, counters, slot, n, fold, host);
}

// ---- frame removal -----------------------------------------------------------------------------
// The mesh is the Delaunay triangulation of the real points and the frame.  Its triangles without
// frame vertices belong to the triangulation of the real points (their circumcircles hold no
// point); what the frame triangles cover has to be triangulated again without the frame.  Every
// triangle there has its three vertices among the real vertices that touch a frame triangle (the
// boundary vertices, B of them), so the triangle left of a directed edge p -> q is found on its own:
// its apex is the boundary vertex left of the edge whose circle through p and q holds no other (the
// minimum of a strict order, ties broken as everywhere).  That is parallel gift wrapping:
//   demand   a directed edge whose left triangle is not known; at first the real edges of the
//            frame triangles, later the far sides of new triangles;
//   apex     one wave looks for it; none: a hull edge;
//   create   one of the demands that found the same triangle claims it, links the sides whose
//            other triangle is known, and its wave goes on with the others.
// Most triangles have a side among the first demands, so the waves' chains are short whatever the
// region's shape: pinches, dangling edges, several components and long straight sides need no
// special case, and one launch does all sets.
// The two demands of an undirected edge {u, v} share an entry e of an open-addressing table.  The
// word own[e] holds, in its low half for u -> v (u < v) and its high half for v -> u, what is left
// of that direction: bit 0 once it is a demand, above it 0 (unknown), 1 + 3 t + k for side k of triangle
// t, or HULL_EDGE.  One atomic OR therefore records a side, lists the other direction and tells what
// was known of it, and no fence orders anything: every link of a new triangle is written by
// whichever of its two sides comes second (or by both, with one value).
// Triangles and demands are those of a planar graph on B vertices: at most 3 B edges.
// Slots: a triangle takes its wave's free slot, that of a dropped frame triangle or a new one.  A wave whose
// triangle was created by another first has a slot left at the end of a demand: at most 2 nt + B new
// slots for nt frame triangles.  Where the capacity has not that many (most vertices on the boundary: 200,000
// points on a curve), hull_tight, all frame triangles' slots are shared and a wave keeps its free slot for its
// next demand.  The new triangles are nt - nf at most (every set loses its frame vertices from the
// hull), so nf + room waves need no more than `room` new slots, whatever they do.
// What bounds it is latency: the dependent reads of an apex and five device-scope atomics of a
// triangle, 5 to 8 us a step.  The boundary stage, against cutting ears of the boundary cycle in
// 16-32 rounds (which needed one simple cycle per set, and left flips to do; sets without one lost
// their frame vertices in 18-58 rounds): 1M uniform points 0.57 -> 0.11 ms, 65,537 0.40 -> 0.08 ms,
// 1,000 (no simple cycle) 0.87 -> 0.06 ms, a batch of 1,024 sets 11.5 -> 1.7 ms.
GA_INLINE bool is_frame_tri(const MeshDev &m, int4 v) { return v.x >= m.n || v.y >= m.n || v.z >= m.n; }
GA_INLINE int frame_vertices(const MeshDev &m, int4 v) { return (v.x >= m.n) + (v.y >= m.n) + (v.z >= m.n); }
GA_INLINE int hull_b(const MeshDev &m, const HullDev &h) { return h.bidx[m.n]; }
// entries of the table for B boundary vertices
GA_INLINE int hull_table(const MeshDev &m, const HullDev &h)
{
    const long long want = 6ll * hull_b(m, h) + 64;
    return (int)(want < h.room ? want : h.room);
}
GA_INLINE bool hull_tight(const MeshDev &m, const HullDev &h)
{
    return m.counters[C_HULL_ROOM] < 2ll * m.counters[C_FTRI] + hull_b(m, h);
}
typedef unsigned long long u64;
#define HULL_LISTED 1u
#define HULL_EDGE 0x7fffffffu
GA_INLINE unsigned hull_value(int t, int k) { return 1u + 3u * (unsigned)t + (unsigned)k; }
GA_INLINE unsigned hull_half(u64 w, int d) { return (unsigned)(w >> (32 * d)); }

// table entry of edge {a, b}, added when it is not there
GA_INLINE int hull_entry(const MeshDev &m, const HullDev &h, int H, int a, int b)
{
    const u64 k = cons_key(a, b);
    unsigned e = (unsigned)(((cons_mix(k) & 0xffffffffull) * (u64)H) >> 32);
    for (int probe = 0; probe < H; probe++) {
        const u64 s = atomicCAS(&h.table[e], 0ull, k);
        if (s == 0 || s == k) return (int)e;
        e = e + 1 == (unsigned)H ? 0u : e + 1;
    }
    atomicOr(m.status, GA_ERR_SCRATCH);   // never: the table holds more entries than there are edges
    return 0;
}

// the frame triangles listed and stamped, their real vertices marked (mark[] zero on entry)
__global__ __launch_bounds__(256) void k_hull_scan(MeshDev m, HullDev h, int op)
{
    const int n = ntri_used(m);
    XCD_STRIDE(b0, n, 1024) {
        unsigned bits = 0;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int t = b0 + j * 256 + (int)threadIdx.x;
            if (t >= n) continue;
            const int4 v = m.tv[t];
            if (v.x == GA_DEAD || !is_frame_tri(m, v)) continue;
            bits |= 1u << j;
            m.stamp[t] = op;
            for (int i = 0; i < 3; i++)
                if (ic(v, i) < m.n) h.mark[ic(v, i)] = 1;
        }
        int k = block_reserve(&m.counters[C_FTRI], __popc(bits));
#pragma unroll
        for (int j = 0; j < 4; j++)
            if ((bits >> j) & 1) h.ftri[k++] = b0 + j * 256 + (int)threadIdx.x;
    }
}

// bidx (the exclusive scan of the marks) numbers the boundary vertices in vertex order, so those of
// a set are consecutive and in spatial order.  Clears the table, places the boundary vertices,
// marks those with a real edge (mark 3), and notes how many slots are unused.
__global__ void k_hull_place(MeshDev m, HullDev h)
{
    if (blockIdx.x == 0 && threadIdx.x == 0) m.counters[C_HULL_ROOM] = m.cap - ntri_used(m);
    const int H = hull_table(m, h), nt = m.counters[C_FTRI];
    GRID_STRIDE(q, nt) {
        const int4 v = m.tv[h.ftri[q]];
        const int one = frame_vertices(m, v) == 1;
#pragma unroll
        for (int i = 0; i < 3; i++) {
            const int a = ic(v, i);
            if (a >= m.n) continue;
            const int k = h.bidx[a];
            h.blist[k] = a;
            h.bpos[k] = m.pos[a];
            if (one) h.mark[a] = 3;
        }
    }
    GRID_STRIDE(e, 2 * H) h.table[e] = 0;   // own follows the keys
}

// The first demands: the real edge of every frame triangle with two real vertices (list: the demand
// and the triangle's slot), with the real triangle across it.  The other frame triangles die here,
// their slots go to the pool (hull_tight: those of all, and the list holds none).  Also the boxes of 64 consecutive boundary vertices each, one wave
// per box.
__global__ __launch_bounds__(256) void k_hull_edges(MeshDev m, HullDev h, int op)
{
    const int H = hull_table(m, h), nt = m.counters[C_FTRI], B = hull_b(m, h);
    const bool tight = hull_tight(m, h);
    u64 *own = h.table + H;
    GRID_STRIDE(qq, nt) {
        const int t = h.ftri[qq];
        const int4 v = m.tv[t];
        const bool one = frame_vertices(m, v) == 1, shared = !one || tight;
        const int k = wave_reserve(&m.counters[C_HULL], one);
        const int kp = wave_reserve(&m.counters[C_HULL_POOL], shared);
        if (shared) {
            h.pool[kp] = t;
            m.tv[t] = make_int4(GA_DEAD, GA_DEAD, GA_DEAD, 0);
        }
        if (!one) continue;
        const int i = v.x >= m.n ? 0 : (v.y >= m.n ? 1 : 2);
        const int p = ic(v, p1(i)), q = ic(v, m1(i)), nb = ic(m.tn[t], i);
        const int e = hull_entry(m, h, H, p, q), d = p < q ? 0 : 1;
        u64 w = (u64)HULL_LISTED << (32 * d);
        if (nb >= 0 && m.stamp[enc_t(nb)] != op) w |= (u64)(hull_value(enc_t(nb), enc_j(nb)) << 1) << (32 * (1 - d));
        atomicOr(&own[e], w);
        h.list[k] = make_int2(2 * e + d, tight ? -1 : t);
    }
    const int lane = threadIdx.x & 63, nw = (gridDim.x * blockDim.x) >> 6;
    for (int g = (blockIdx.x * blockDim.x + threadIdx.x) >> 6; 64 * g < B; g += nw) {
        const double2 X = h.bpos[min(64 * g + lane, B - 1)];
        double lx = X.x, ly = X.y, hx = X.x, hy = X.y;
        for (int d = 32; d > 0; d >>= 1) {
            lx = fmin(lx, __shfl_xor(lx, d, 64)); ly = fmin(ly, __shfl_xor(ly, d, 64));
            hx = fmax(hx, __shfl_xor(hx, d, 64)); hy = fmax(hy, __shfl_xor(hy, d, 64));
        }
        if (lane == 0) h.bbox[g] = HullBox{lx, ly, hx, hy};
    }
}

// The boundary vertices [b0, b1) of a set, and a power of two that brings the differences of its
// coordinates to 2^15 at most.  The searches below decide in floating point what can be left out, by products
// of up to three differences: without it these lose their bits below coordinates of 1e-103, and are
// infinite above 1e154, where the order of the apexes (t) becomes NaN.  What is still too small (vertices
// that lie 1e-100 of the set's size and less apart) is not left out.
struct HullSet {
    int b0, b1;
    double s;
};
#define HULL_TINY 1e-290   // above what is lost to underflow in scaled coordinates
__device__ HullSet hull_set(const MeshDev &m, const HullDev &h, int v)
{
    const SetDesc &sd = m.sets[m.vset[v]];
    const int e = -ilogb(sd.scale);
    return HullSet{h.bidx[sd.poff], h.bidx[sd.poff + sd.n], ldexp(1.0, e < 1023 ? e : 1023)};
}

// squared distances to v: true when a is nearer than b
__device__ __noinline__ bool hull_nearer(double2 v, double2 a, double2 b, double sc, int *status)
{
    const double ax = (a.x - v.x) * sc, ay = (a.y - v.y) * sc, bx = (b.x - v.x) * sc, by = (b.y - v.y) * sc;
    const double da = ax * ax + ay * ay, db = bx * bx + by * by, eb = 8.0 * GA_EPS * (da + db) + HULL_TINY;
    if (da - db < -eb) return true;
    if (da - db > eb) return false;
    // |a - v|^2 - |b - v|^2 exactly
    int ovf = 0;
    const double c[6] = {v.x, v.y, a.x, a.y, b.x, b.y};
    const int s = min_ulp_exp(c, 6);
    BigInt<12> V, A, B, x, sum;
    bi_zero(sum);
    for (int k = 0; k < 2; k++) {
        bi_from_double(V, c[k], s, &ovf);
        bi_from_double(A, c[2 + k], s, &ovf);
        bi_from_double(B, c[4 + k], s, &ovf);
        bi_sub(A, A, V, &ovf);
        bi_sub(B, B, V, &ovf);
        bi_mul(x, A, A, &ovf);
        bi_add(sum, sum, x, &ovf);
        bi_mul(x, B, B, &ovf);
        bi_sub(sum, sum, x, &ovf);
    }
    if (ovf) atomicOr(status, GA_ERR_EXACT_OVERFLOW);
    return bi_sign(sum) < 0;
}

// the boundary vertex of the set nearest to its position k (one wave; -1: there is no other)
GA_INLINE int hull_nearest(const MeshDev &m, const HullDev &h, int k, HullSet set, int lane)
{
    const double2 P = h.bpos[k];
    int best = -1;
    for (int j = set.b0 + lane; j < set.b1; j += 64)
        if (j != k && (best < 0 || hull_nearer(P, h.bpos[j], h.bpos[best], set.s, m.status))) best = j;
    for (int d = 32; d > 0; d >>= 1) {
        const int o = __shfl_xor(best, d, 64);
        if (o >= 0 && (best < 0 || hull_nearer(P, h.bpos[o], h.bpos[best], set.s, m.status))) best = o;
    }
    return best < 0 ? -1 : h.blist[best];
}

// Incircle sign of boundary vertices: the search asks for many vertices near one circle (along an arc, for 64
// vertices of every box), and the exact test keeps its numbers in scratch memory: boundary stage of 30,000
// points on half a circle 124 ms, 14 with the pairs of doubles before it; 200,000 points 196 ms.
__device__ __noinline__ int hull_incircle_dd(double2 a, double2 b, double2 c, double2 d, double sc)
{
    return incircle_dd(a, b, c, d, sc);
}
GA_INLINE int hull_incircle(const MeshDev &m, double2 a, double2 b, double2 c, double2 d, int ia, int ib, int ic_, int id,
                            double sc)
{
    int s = incircle_filter(a, b, c, d);
    if (s == 0) s = hull_incircle_dd(a, b, c, d, sc);
    return s != 0 ? s : incircle_at(m, a, b, c, d, ia, ib, ic_, id);
}

// a candidate apex of p -> q
struct HullBest {
    int v;        // -1: none
    double2 X;
};

// The wave's best c (the same in all lanes) against the boundary positions 64 g + lane of the set:
// replaced by a vertex left of p -> q and inside its circle until no lane has one.  The
// next to try is the one that sees the edge under the largest angle (in floating point: it only
// decides how often the loop runs, mostly once).
GA_INLINE void hull_chunk(const MeshDev &m, const HullDev &h, double2 P, double2 Q, int p, int q, int g, HullSet set,
                          int lane, HullBest &c)
{
    const int j = 64 * g + lane;
    const bool in = j >= set.b0 && j < set.b1;
    const double2 X = in ? h.bpos[j] : P;
    const int x = in ? h.blist[j] : p;
    int o = orient_filter(P, Q, X);
    // p, q themselves and points on one axis-parallel line with them are exactly collinear
    if (o == 0 && x != p && x != q && !(P.x == Q.x && Q.x == X.x) && !(P.y == Q.y && Q.y == X.y)) {
        o = orient_diff(P, Q, X);   // (a search along 20,000 points on a sloped line: half the time)
        if (o == 2) o = orient_dev(m, P, Q, X);
    }
    bool better = o > 0 && x != p && x != q;
    double t = INFINITY;
    if (better) {
        const double ax = (P.x - X.x) * set.s, ay = (P.y - X.y) * set.s;
        const double bx = (Q.x - X.x) * set.s, by = (Q.y - X.y) * set.s;
        const double cr = ax * by - ay * bx, dot = ax * bx + ay * by;
        t = cr > 0.0 ? dot / cr : (dot < 0.0 ? -INFINITY : INFINITY);
        if (c.v >= 0) better = x != c.v && hull_incircle(m, P, Q, c.X, X, p, q, c.v, x, set.s) > 0;
    }
    while (__any(better)) {
        double mt = better ? t : INFINITY;
        for (int d = 32; d > 0; d >>= 1) mt = fmin(mt, __shfl_xor(mt, d, 64));
        const int k = __ffsll((long long)__ballot(better && t <= mt)) - 1;
        c = HullBest{__shfl(x, k, 64), make_double2(__shfl(X.x, k, 64), __shfl(X.y, k, 64))};
        if (better) better = x != c.v && hull_incircle(m, P, Q, c.X, X, p, q, c.v, x, set.s) > 0;
    }
}

// p -> q lies on the line of a hull edge found before (h.lines: some whose search took more than 16 boxes;
// lane k tests line k), in its direction: then it is a hull edge as well.  Without that, every edge of a long
// straight side looks at every box that the side passes through (two sloped sides of 30,000 points each: 127 ms, 2.4
// with it).
__device__ bool hull_on_line(const MeshDev &m, const HullDev &h, int p, int q, double2 P, double2 Q, HullSet set, int lane)
{
    bool on = false;
    if (lane < HULL_LINES) {
        const unsigned long long e = __hip_atomic_load(&h.lines[lane], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const int a = (int)(e >> 32), b = (int)(e & 0xffffffffull);
        if (a != b && h.bidx[a] >= set.b0 && h.bidx[a] < set.b1) {
            const double2 A = m.pos[a], B = m.pos[b];
            on = (A.x < B.x) == (P.x < Q.x) && (A.x > B.x) == (P.x > Q.x) && (A.y < B.y) == (P.y < Q.y) &&
                 (A.y > B.y) == (P.y > Q.y) && orient_dev(m, A, B, P) == 0 && orient_dev(m, A, B, Q) == 0;
        }
    }
    return __any(on);
}

// The apex of p -> q among the boundary vertices of its set (one wave; -1: none).  First
// the vertices numbered next to p and q, which gives a circle near the final one; then the
// boxes, 64 at a time: a box can hold a better apex only if it reaches left of the edge and into
// the circle, which leaves one to three of B / 64.  (Every vertex tested, in steps of 64, took
// 51 us per launch at B = 2,500, one dependent read after another.)  Both box tests keep a margin
// far above their rounding; a circle too flat or too small for that is not used.
__device__ int hull_apex(const MeshDev &m, const HullDev &h, int p, int q, HullSet set, int lane)
{
    const double sc = set.s;

    const double2 P = m.pos[p], Q = m.pos[q];
    const int gp = h.bidx[p] >> 6, gq = h.bidx[q] >> 6;
    HullBest c{-1, P};
    hull_chunk(m, h, P, Q, p, q, gp, set, lane, c);
    if (gq != gp) hull_chunk(m, h, P, Q, p, q, gq, set, lane, c);
    const double ux = (Q.x - P.x) * sc, uy = (Q.y - P.y) * sc;
    const int g1 = (set.b1 - 1) >> 6;
    bool asked = !h.lines;
    for (int gb = set.b0 >> 6; gb <= g1; gb += 64) {
        const int g = gb + lane;
        const bool in = g <= g1 && g != gp && g != gq;
        const HullBox bx = h.bbox[min(g, g1)];
        // largest cross product (Q - P) x (X - P) over the box, at its corner (cx, cy); exactly zero when that
        // lies on an axis-parallel line with p and q
        const double cx = uy > 0 ? bx.lx : bx.hx, cy = ux > 0 ? bx.hy : bx.ly;
        const double l = ux * ((cy - P.y) * sc), r = uy * ((cx - P.x) * sc);
        const bool flat = (P.x == Q.x && cx == P.x) || (P.y == Q.y && cy == P.y);
        // (a box with vertices of another set may be so large that this is NaN: it stays)
        const bool left = in && !flat && !(l - r < -1e-14 * (fabs(l) + fabs(r)) - HULL_TINY);
        unsigned long long todo = __ballot(left);
        if (!asked && c.v < 0 && __popcll(todo) > 16) {
            asked = true;
            if (hull_on_line(m, h, p, q, P, Q, set, lane)) return -1;
        }
        while (todo) {
            if (c.v >= 0) {
                // circle of (P, Q, C): centre P + (ox, oy)
                const double vx = (c.X.x - P.x) * sc, vy = (c.X.y - P.y) * sc;
                const double a = ux * vy, b = uy * vx, cr = a - b;
                // (cr > 1e-200: the radius is above 1e-101, what the products below lose, times f, below 1e-118)
                if (cr > 1e-6 * (fabs(a) + fabs(b)) && cr > 1e-200) {
                    const double uu = ux * ux + uy * uy, vv = vx * vx + vy * vy, f = 0.5 / cr;
                    const double ox = f * (vy * uu - uy * vv), oy = f * (ux * vv - vx * uu);
                    const double dx = fmax(fmax((bx.lx - P.x) * sc - ox, ox - (bx.hx - P.x) * sc), 0.0);
                    const double dy = fmax(fmax((bx.ly - P.y) * sc - oy, oy - (bx.hy - P.y) * sc), 0.0);
                    const double rad = sqrt(ox * ox + oy * oy);
                    // the relative error of f and of the differences, the centre's cancellation error
                    const double reach = rad * (1.0 + 1e-8) +
                                         1e-14 * f * ((fabs(vx) + fabs(vy)) * uu + (fabs(ux) + fabs(uy)) * vv);
                    const bool out = dx * dx + dy * dy > reach * reach;
                    todo &= ~__ballot(out);
                    if (!todo) break;
                }
            }
            const int k = __ffsll((long long)todo) - 1;
            todo &= todo - 1;
            hull_chunk(m, h, P, Q, p, q, gb + k, set, lane, c);
        }
    }
    if (asked && c.v < 0 && h.lines && lane == 0)
        __hip_atomic_store(&h.lines[p % HULL_LINES], (unsigned long long)p << 32 | (unsigned)q, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
    return c.v;
}

// Creates the triangle (p, q, c) unless another demand did, in *slot when the wave has one (then
// -1), else in one from the pool (its share of it, or any: all) or a new one; pushes the far sides that nothing is known of on the
// wave's stack (next[] links the demands, *head the first).  One wave; lanes 0, 1 and 2 take a side each.
__device__ void hull_create(const MeshDev &m, const HullDev &h, int H, int it0, int p, int q, int c, bool all, int lane,
                            int *slot, int *head)
{
    u64 *own = h.table + H;
    // the sides from the smallest vertex a; the wave that sets the left of a -> b creates the triangle
    const int r = p < q ? (p < c ? 0 : 2) : (q < c ? 1 : 2);
    const int a = r == 0 ? p : (r == 1 ? q : c), b = r == 0 ? q : (r == 1 ? c : p), d = r == 0 ? c : (r == 1 ? p : q);
    const int su = lane == 0 ? a : (lane == 1 ? b : d), sv = lane == 0 ? b : (lane == 1 ? d : a);
    const int k = lane == 0 ? 2 : (lane == 1 ? 0 : 1);   // the side lies opposite vertex k of (a, b, d)
    int it = 0, T = *slot;
    if (lane < 3) it = 2 * hull_entry(m, h, H, su, sv) + (su < sv ? 0 : 1);
    if (T < 0 && lane == 0) {
        // the pool's shares are taken one by one, so that no counter serves all waves
        int s = (int)((blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6)) % HULL_SHARES);
        for (int u = all ? HULL_SHARES : 1; u > 0 && T < 0; u--, s = (s + 1) % HULL_SHARES) {
            const int x = s + HULL_SHARES * atomicAdd(&h.share[s * HULL_SHARE_INTS], 1);
            if (x < m.counters[C_HULL_POOL]) T = h.pool[x];
        }
        if (T < 0) T = atomicAdd(m.ntri, 1);
    }
    T = __shfl(T, 0, 64);
    if (T >= m.cap) {
        if (lane == 0) atomicOr(m.status, GA_ERR_CAPACITY);
        return;
    }
    *slot = T;
    const unsigned val = hull_value(T, k) << 1;
    bool won = false;
    if (lane == 0) {
        unsigned *half = (unsigned *)&own[it >> 1];   // a < b: the low half
        unsigned w = it == it0 ? HULL_LISTED : 0u;
        while (w <= HULL_LISTED) {
            const unsigned seen = atomicCAS(half, w, val | w);
            if (seen == w) { won = true; break; }
            w = seen;
        }
    }
    if (!__shfl((int)won, 0, 64)) return;
    *slot = -1;
    bool more = false;
    if (lane < 3) {
        const int dir = it & 1;
        const u64 w = (lane == 0 ? 0ull : (u64)val << (32 * dir)) | ((u64)HULL_LISTED << (32 * (1 - dir)));
        const unsigned o = hull_half(atomicOr(&own[it >> 1], w), 1 - dir);
        const unsigned ov = o >> 1;
        if (ov == HULL_EDGE) set_link(m, T, k, -1);
        else if (ov) bond(m, T, k, enc((int)((ov - 1) / 3u), (int)((ov - 1) % 3u)));
        else more = o == 0;   // this wave has listed it
    }
    if (lane == 0) m.tv[T] = make_int4(a, b, d, 0);
    const unsigned long long mb = __ballot(more);
    for (int s = 0; s < 3; s++) {
        if (!((mb >> s) & 1)) continue;
        const int x = __shfl(it, s, 64) ^ 1;
        if (lane == 0) h.next[x] = *head;
        *head = x;
    }
}

// Drops the frame vertices and the frame triangles left, and fills what they covered: one wave per
// first demand (with its frame triangle's slot) and per boundary vertex without a real edge.  For such
// a vertex the edge to its nearest boundary vertex is a Delaunay edge (the circle on it as diameter is
// empty) with nothing known on either side.
__global__ __launch_bounds__(256) void k_hull_fill(MeshDev m, HullDev h)
{
    const int H = hull_table(m, h), nd = m.counters[C_HULL], B = hull_b(m, h);
    u64 *own = h.table + H;
    GRID_STRIDE(k, m.V - m.n) {
        const int f = m.n + k;
        if (m.vstate[f] == VS_IN_MESH) m.vstate[f] = VS_REMOVED;
        m.vt[f] = -1;
    }
    const bool tight = hull_tight(m, h);
    const int lane = threadIdx.x & 63, all = (int)((gridDim.x * blockDim.x) >> 6);
    const int nw = tight ? min(all, m.V - m.n + m.counters[C_HULL_ROOM]) : all;
    const int w0 = (int)((blockIdx.x * blockDim.x + threadIdx.x) >> 6);
    int slot = -1;
    for (int i = w0 < nw ? w0 : nd + B; i < nd + B; i += nw) {
        int head = -1;
        HullSet set;
        if (i < nd) {
            const int2 f = h.list[i];
            head = f.x;
            if (!tight) slot = f.y;
            if (lane == 0) h.next[head] = -1;
            set = hull_set(m, h, (int)((h.table[head >> 1] - 1) >> 32));
        } else {
            const int v = h.blist[i - nd];
            if (h.mark[v] == 3) continue;
            set = hull_set(m, h, v);
            const int w = hull_nearest(m, h, i - nd, set, lane);
            if (w < 0) continue;
            int e = 0;
            u64 old = 0;
            if (lane == 0) {
                e = hull_entry(m, h, H, v, w);
                old = atomicOr(&own[e], (u64)HULL_LISTED << 32 | HULL_LISTED);
            }
            e = __shfl(e, 0, 64);
            old = __shfl(old, 0, 64);
            for (int d = 0; d < 2; d++)
                if (hull_half(old, d) == 0) {
                    if (lane == 0) h.next[2 * e + d] = head;
                    head = 2 * e + d;
                }
        }
        while (head >= 0) {
            const int it = head;
            int nx = 0, known = 0;
            u64 key = 0;
            if (lane == 0) {
                nx = h.next[it];
                const u64 w = __hip_atomic_load(&own[it >> 1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                known = hull_half(w, it & 1) > HULL_LISTED;   // found from another side
                key = __hip_atomic_load(&h.table[it >> 1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) - 1;
            }
            head = __shfl(nx, 0, 64);
            if (__shfl(known, 0, 64)) continue;
            key = __shfl(key, 0, 64);
            const int lo = (int)(key >> 32), hi = (int)(key & 0xffffffffull);
            const int p = it & 1 ? hi : lo, q = it & 1 ? lo : hi;
            const int c = hull_apex(m, h, p, q, set, lane);
            if (c >= 0) {
                hull_create(m, h, H, it, p, q, c, tight, lane, &slot, &head);
                continue;
            }
            if (lane == 0) {
                const int d = it & 1;
                const unsigned ov = hull_half(atomicOr(&own[it >> 1], (u64)(HULL_EDGE << 1) << (32 * d)), 1 - d) >> 1;
                if (ov && ov != HULL_EDGE) set_link(m, (int)((ov - 1) / 3u), (int)((ov - 1) % 3u), -1);
            }
        }
        if (tight) continue;
        if (slot >= 0 && lane == 0) m.tv[slot] = make_int4(GA_DEAD, GA_DEAD, GA_DEAD, 0);
        slot = -1;
    }
    if (slot >= 0 && lane == 0) m.tv[slot] = make_int4(GA_DEAD, GA_DEAD, GA_DEAD, 0);
}

void launch_hull(MeshDev &m, const HullDev &h, int op, void *scan_tmp, hipStream_t st)
{
    GA_LAUNCH(k_hull_scan, dim3(FIXED_GRID), dim3(256), 0, st, m, h, op);
    launch_exclusive_scan(h.mark, h.bidx, (size_t)m.n + 1, scan_tmp, st);
    GA_LAUNCH(k_hull_place, dim3(FIXED_GRID), dim3(256), 0, st, m, h);
    GA_LAUNCH(k_hull_edges, dim3(FIXED_GRID), dim3(256), 0, st, m, h, op);
    GA_LAUNCH(k_hull_fill, dim3(FIXED_GRID), dim3(256), 0, st, m, h);
}

// ---- canonical output ----------------------------------------------------------------------------
// Output order: (v0, v1, v2) of input indices with v0 the smallest vertex; input indices of the sets
// of a batch are consecutive ranges in set order, so this is also set order.  Every directed edge
// belongs to one triangle, so (v0, v1) alone is unique: the key is v0 << B | v1 (indices below 2^B),
// sorted on its low 2B bits.  Dead slots get all ones there, above every live key (v0 <= n - 3).
__global__ void k_canon_keys(MeshDev m, unsigned long long *keys, int *vals, int *rot, int B, int count)
{
    int n = ntri_used(m);
    int alive = 0;
    GRID_STRIDE(t, n) {
        int4 v = m.tv[t];
        vals[t] = t;
        if (v.x == GA_DEAD) { keys[t] = ~0ull; rot[t] = 0; continue; }
        alive++;
        int4 o = make_int4(oid(m, v.x), oid(m, v.y), oid(m, v.z), 0);   // input indices
        int r = 0;
        if (o.y < ic(o, r)) r = 1;
        if (o.z < ic(o, r)) r = 2;
        rot[t] = r;
        unsigned long long a = (unsigned)ic(o, r), b = (unsigned)ic(o, (r + 1) % 3);
        keys[t] = (a << B) | b;
    }
    if (count) stat_add_full(m.stats, C_RECON_TRIS, alive);
}

void launch_canon_keys(MeshDev &m, unsigned long long *keys, int *vals, int *rot, int B, bool count, hipStream_t st)
{
    GA_LAUNCH(k_canon_keys, dim3(FIXED_GRID), dim3(256), 0, st, m, keys, vals, rot, B, count ? 1 : 0);
}

// 32-bit keys (indices below 2^B, B <= CANON_KEY32_BITS): v0 in the top B bits, then the top
// W = min(B, 32 - B) bits of v1 - v0, which is below the number of points of the set: at most four
// radix passes (the whole pair in 64-bit keys takes six at B = 22 and 24: the passes of 4M points 458 us
// against 235, of 1,024 sets 1,170 against 560).  They order the triangles up to runs of equal keys
// (the same v0 and close v1), which k_canon_newid orders.  v1[t] keeps v1 for it.  Dead slots get
// all ones, above every live key (v0 <= n - 3).
__global__ void k_canon_keys32(MeshDev m, unsigned *keys, unsigned *v1s, int *vals, int *rot, int B)
{
    int n = ntri_used(m);
    int alive = 0;
    const int W = min(B, 32 - B);
    GRID_STRIDE(t, n) {
        int4 v = m.tv[t];
        vals[t] = t;
        if (v.x == GA_DEAD) { keys[t] = 0xffffffffu; rot[t] = 0; continue; }
        alive++;
        int4 o = make_int4(oid(m, v.x), oid(m, v.y), oid(m, v.z), 0);   // input indices
        int r = 0;
        if (o.y < ic(o, r)) r = 1;
        if (o.z < ic(o, r)) r = 2;
        rot[t] = r;
        const unsigned a = (unsigned)ic(o, r), b = (unsigned)ic(o, (r + 1) % 3);
        int np = m.n;
        if (m.nsets > 1) {
            const int set = m.vset[v.x];
            np = (set + 1 < m.nsets ? m.sets[set + 1].poff : m.n) - m.sets[set].poff;
        }
        const int drop = max(32 - __clz(np - 1) - W, 0);   // low bits of v1 - v0 left out
        keys[t] = (a << W) | ((b - a) >> drop);
        v1s[t] = b;
    }
    stat_add_full(m.stats, C_RECON_TRIS, alive);
}

void launch_canon_keys32(MeshDev &m, unsigned *keys, unsigned *v1s, int *vals, int *rot, int B, hipStream_t st)
{
    GA_LAUNCH(k_canon_keys32, dim3(FIXED_GRID), dim3(256), 0, st, m, keys, v1s, vals, rot, B);
}

// newid[slot] = output position << 2 | rotation of the slot's triangle: one gather per neighbour
// in k_canon_emit.  With 32-bit keys (skey, v1s non-null) every triangle of a run of equal sorted
// keys counts those with a smaller v1; out[] gets the final order.  Runs are mostly short.  Around one vertex
// with all others as neighbours they have up to 2^(2B - 32) entries (256 at B = 20, 2^16 at 24), and counting is
// quadratic: a run of more than CANON_RUN entries is left as it is and reported, and the host orders by whole
// keys instead (4.2M points, one with 400,000 neighbours: canonical stage 179 ms with counting alone, 2.3 now;
// 1.1M points, one with 1,000 neighbours, where counting is still the cheaper: 0.49 and 0.81).
#define CANON_RUN 512
__global__ void k_canon_newid(const int *order, const unsigned *skey, const unsigned *v1s, const int *rot, const int *dF,
                              int *newid, int *out, int *long_run)
{
    int F = *dF;
    GRID_STRIDE(r, F) {
        const int s = order[r];
        int at = r;
        if (skey) {
            const unsigned key = skey[r];
            const bool before = r > 0 && skey[r - 1] == key, after = r + 1 < F && skey[r + 1] == key;
            if (before || after) {
                const unsigned v = v1s[s];
                // others of the run that are looked at; none when it is seen to be too long from here
                const bool far = (r + CANON_RUN < F && skey[r + CANON_RUN] == key) || (r >= CANON_RUN && skey[r - CANON_RUN] == key);
                int room = far ? 0 : CANON_RUN;
                for (int j = r - 1; j >= 0 && room > 0 && skey[j] == key; j--, room--) at -= v1s[order[j]] > v;
                for (int j = r + 1; j < F && room > 0 && skey[j] == key; j++, room--) at += v1s[order[j]] < v;
                if (room == 0) {   // (for every triangle of the run: the order stays a permutation)
                    at = r;
                    if (!before) *long_run = 1;
                }
            }
            out[at] = s;
        }
        newid[s] = (at << 2) | rot[s];
    }
}

// out9 holds global vertex ids and global triangle positions.  The slots are in spatial order and the
// output is in the order of the input indices, so one of the two sides is scattered whatever the
// order of the work: k_canon_records makes the six words of a slot's record in slot order (its
// neighbours' positions and its vertices' ids lie close together there), and k_canon_emit, one thread
// per output record, gathers them, so that neighbouring lanes write whole records (gathering vertices,
// links, positions and ids per output record instead took 565 us at 4M points, this 356; 129 and 84 at
// 1M).  A batch's sets are small enough that the gathers of a set stay in its L2: there
// k_canon_emit_sets makes the records on the way (1,024 sets: 1,354 us, in two steps 1,608).
__global__ __launch_bounds__(256) void k_canon_records(MeshDev m, const int *newid, int2 *rec)
{
    const int n = ntri_used(m);
    GRID_STRIDE(t, n) {
        const int4 v = m.tv[t];
        if (v.x == GA_DEAD) continue;
        const int4 nb = m.tn[t];
        const int ro = newid[t] & 3;
        int w[6];
#pragma unroll
        for (int i = 0; i < 3; i++) {
            const int si = (i + ro) % 3;
            w[3 + i] = oid(m, ic(v, si));
            const int e = ic(nb, si);
            w[i] = -1;
            if (e >= 0) {
                const int nu = newid[enc_t(e)];
                w[i] = enc(nu >> 2, (enc_j(e) - (nu & 3) + 3) % 3);
            }
        }
#pragma unroll
        for (int i = 0; i < 3; i++) rec[3 * (size_t)t + i] = make_int2(w[2 * i], w[2 * i + 1]);
    }
}

__global__ __launch_bounds__(256) void k_canon_emit(const int *order, const int2 *rec, const int *dF, int *out9)
{
    const int F = *dF;
    for (int r = blockIdx.x * 256 + threadIdx.x; r < F; r += gridDim.x * 256) {
        const int2 *w = rec + 3 * (size_t)order[r];
        const int2 a = w[0], b = w[1], c = w[2];
        int *o = out9 + (size_t)r * 9;
        o[0] = a.x; o[1] = a.y; o[2] = b.x;
        o[3] = b.y; o[4] = c.x; o[5] = c.y;
        o[6] = 0; o[7] = 0; o[8] = 0;
    }
}

// rset[r] = set of output triangle r, for k_canon_set_first
__global__ void k_canon_emit_sets(MeshDev m, const int *order, const int *newid, const int *dF, int *out9, int *rset)
{
    const int F = *dF;
    GRID_STRIDE(r, F) {
        const int s = order[r];
        const int4 v = m.tv[s];
        const int ro = newid[s] & 3;
        const int4 nb = m.tn[s];
        int rec[9];
#pragma unroll
        for (int i = 0; i < 3; i++) {
            const int si = (i + ro) % 3;
            rec[3 + i] = oid(m, ic(v, si));
            const int e = ic(nb, si);
            if (e < 0) rec[i] = -1;
            else {
                const int nu = newid[enc_t(e)];
                rec[i] = enc(nu >> 2, (enc_j(e) - (nu & 3) + 3) % 3);
            }
            rec[6 + i] = 0;
        }
        int *o = out9 + (size_t)r * 9;
#pragma unroll
        for (int i = 0; i < 9; i++) o[i] = rec[i];
        rset[r] = m.vset[v.x];
    }
}

// set_first[s] = first output triangle of set s (left at -1 for a set without triangles)
__global__ void k_canon_set_first(MeshDev m, const int *rset, const int *dF, int *set_first)
{
    int F = *dF;
    GRID_STRIDE(r, F) {
        int set = rset[r];
        if (r == 0 || rset[r - 1] != set) set_first[set] = r;
    }
}

void launch_canon_emit(MeshDev &m, const int *order, const unsigned *skey, const unsigned *v1s, int *out, const int *rot,
                       int *newid, int2 *rec, const int *dF, int *out9, int *set_first, int *rset, hipStream_t st)
{
    GA_LAUNCH(k_canon_newid, dim3(FIXED_GRID), dim3(256), 0, st, order, skey, v1s, rot, dF, newid, out,
              m.counters + C_LONG_RUN);
    const int *sorted = skey ? out : order;
    if (m.nsets == 1) {   // (its first triangle is triangle 0)
        GA_LAUNCH(k_canon_records, dim3(FIXED_GRID), dim3(256), 0, st, m, (const int *)newid, rec);
        GA_LAUNCH(k_canon_emit, dim3(FIXED_GRID), dim3(256), 0, st, sorted, (const int2 *)rec, dF, out9);
        return;
    }
    GA_LAUNCH(k_canon_emit_sets, dim3(FIXED_GRID), dim3(256), 0, st, m, sorted, (const int *)newid, dF, out9, rset);
    launch_fill_i32(set_first, -1, (size_t)m.nsets, st);
    GA_LAUNCH(k_canon_set_first, dim3(FIXED_GRID), dim3(256), 0, st, m, (const int *)rset, dF, set_first);
}

// ---- constrained DT ---------------------------------------------------------------------------
// Constraint edges go into the finished DT by cavity retriangulation.  A constraint (a, b) walks
// from a to b and collects the triangles it crosses (its cavity) with the chains of vertices
// left and right of it.  Cavities claim their slots; every constraint that holds all of its slots
// replaces its cavity by triangulations of the two pseudo-polygons on either side of the new edge.
// Each is built by taking the chain vertex whose circle through the base edge holds no other chain
// vertex (tie-broken incircle, the order the flip pass uses) and recursing on both sides.  A cavity
// of K triangles has K + 2 vertices, so the new triangles reuse its K slots.  A constrained flip
// pass afterwards (k_flip_test skips constraint edges) makes every other edge locally Delaunay.
// The reference inserts by parallel flips instead (Cuda/cudaConstraint.cu:143-939) and marks the
// constraint edges for its flip pass (Cuda/cudaFlipping.cu:111-220); the result, the constrained
// DT, is unique under the tie-break.

__global__ void k_cons_inv(MeshDev m, int *inv)
{
    GRID_STRIDE(v, m.n) inv[m.perm[v]] = v;
}

__global__ void k_cons_map(MeshDev m, const int2 *cin, int nc, const int *inv, int2 *cv, int *done,
                           unsigned long long *chash, int chmask)
{
    GRID_STRIDE(c, nc) {
        int a = inv[cin[c].x], b = inv[cin[c].y];
        cv[c] = make_int2(a, b);
        done[c] = 0;
        if (m.vstate[a] == VS_DUP || m.vstate[b] == VS_DUP) {
            atomicOr(m.status, GA_ERR_CONS_DUP);
            done[c] = 1;
            continue;
        }
        unsigned long long k = cons_key(a, b);
        for (unsigned long long h = cons_mix(k);; h++) {
            unsigned long long prev = atomicCAS(&chash[h & (unsigned long long)chmask], 0ull, k);
            if (prev == 0 || prev == k) break;
        }
    }
}

// every vertex's anchor triangle from the live slots (frame removal leaves some anchors stale)
__global__ void k_cons_vt(MeshDev m)
{
    int n = ntri_used(m);
    GRID_STRIDE(t, n) {
        int4 tt = m.tv[t];
        if (tt.x == GA_DEAD) continue;
        m.vt[tt.x] = t;
        m.vt[tt.y] = t;
        m.vt[tt.z] = t;
    }
}

// ints of a cavity region of K triangles: K, ml, mr, pad; slots[K]; Lx[K + 2]; Rx[K + 2];
// lb[K + 1]; rb[K + 1]; ol[K + 1]; orr[K + 1]; stack[3 (K + 2)]
GA_INLINE int cons_region(int K) { return 10 * K + 18; }

struct ConsRegion {
    int *hdr, *slots, *Lx, *Rx, *lb, *rb, *ol, *orr, *stk;
    __device__ ConsRegion(int *r, int K)
    {
        hdr = r;
        slots = r + 4;
        Lx = slots + K;
        Rx = Lx + K + 2;
        lb = Rx + K + 2;
        rb = lb + K + 1;
        ol = rb + K + 1;
        orr = ol + K + 1;
        stk = orr + K + 1;
    }
};

// Walk of constraint (a, b).  Returns the cavity size K >= 1, 0 when the edge exists already, -1
// on an error (status set).  With REC the cavity is written to the region sized for Kc triangles:
// slots in walk order; Lx = a, left chain, b and Rx = a, right chain, b; lb[i] / rb[i] = the
// cavity side (t << 2 | j) on the boundary edge between Lx[i], Lx[i + 1] / Rx[i], Rx[i + 1].
template <bool REC>
__device__ int cons_walk(const MeshDev &m, int a, int b, ConsRegion *R, int Kc)
{
    double2 A = m.pos[a], B = m.pos[b];
    int t0 = m.vt[a], t = -1, k = 0;
    if (t0 < 0 || t0 >= m.cap) {
        atomicOr(m.status, GA_ERR_CONS_WALK);
        return -1;
    }
    // the triangle (a, p, q) of a's star with b strictly inside its angle at a
    for (int dir = 0; dir < 2 && t < 0; dir++) {
        int s = t0;
        for (int guard = 0; guard < 1000000; guard++) {
            int4 tt = m.tv[s];
            int ka = tt.x == a ? 0 : (tt.y == a ? 1 : 2);
            int p = ic(tt, p1(ka)), q = ic(tt, m1(ka));
            if (p == b || q == b) return 0;
            double2 P = m.pos[p], Q = m.pos[q];
            int op = orient_dev(m, A, P, B), oq = orient_dev(m, A, Q, B);
            // a vertex on the ray from a towards b lies inside the segment (b itself is not on
            // an edge of a's star)
            if ((op == 0 && (P.x - A.x) * (B.x - A.x) + (P.y - A.y) * (B.y - A.y) > 0) ||
                (oq == 0 && (Q.x - A.x) * (B.x - A.x) + (Q.y - A.y) * (B.y - A.y) > 0)) {
                atomicOr(m.status, GA_ERR_CONS_POINT);
                return -1;
            }
            if (op > 0 && oq < 0) {
                t = s;
                k = ka;
                break;
            }
            // counter-clockwise: across (a, q), the side opposite p; clockwise: across (a, p)
            int e = ic(m.tn[s], dir == 0 ? p1(ka) : m1(ka));
            if (e < 0) break;
            s = enc_t(e);
            if (s == t0) break;
        }
    }
    if (t < 0) {
        atomicOr(m.status, GA_ERR_CONS_WALK);
        return -1;
    }
    int4 tt = m.tv[t];
    int p = ic(tt, p1(k)), q = ic(tt, m1(k));   // p right of a -> b, q left
    int K = 1, ml = 1, mr = 1;
    if (REC) {
        R->slots[0] = t;
        R->Lx[0] = a; R->Lx[1] = q;
        R->Rx[0] = a; R->Rx[1] = p;
        R->lb[0] = enc(t, p1(k));   // edge (q, a)
        R->rb[0] = enc(t, m1(k));   // edge (a, p)
    }
    int cur = t, ex = k;
    for (int guard = 0; guard < m.cap; guard++) {
        int e = ic(m.tn[cur], ex);
        if (e < 0) break;
        int u = enc_t(e), j = enc_j(e);
        int4 ut = m.tv[u];
        // entered across (r1, r2): r1 left of a -> b, r2 right; w is the far vertex
        int w = ic(ut, j), r1 = ic(ut, p1(j)), r2 = ic(ut, m1(j));
        if (cons_has(m, r1, r2)) {
            atomicOr(m.status, GA_ERR_CONS_CROSS);
            return -1;
        }
        if (REC && K >= Kc) break;   // the mesh changed since the count: report below
        if (REC) R->slots[K] = u;
        K++;
        if (w == b) {
            if (REC) {
                R->lb[ml] = enc(u, m1(j));   // edge (r1, b)
                R->rb[mr] = enc(u, p1(j));   // edge (b, r2)
                R->Lx[ml + 1] = b;
                R->Rx[mr + 1] = b;
                R->hdr[0] = K; R->hdr[1] = ml; R->hdr[2] = mr;
            }
            return K;
        }
        int o = orient_dev(m, A, B, m.pos[w]);
        if (o == 0) {   // w is on the segment (the walk has not reached b)
            atomicOr(m.status, GA_ERR_CONS_POINT);
            return -1;
        }
        if (o > 0) {   // w joins the left chain; leave across (w, r2)
            if (REC) { R->lb[ml] = enc(u, m1(j)); R->Lx[ml + 1] = w; }
            ml++;
            ex = p1(j);
        } else {       // w joins the right chain; leave across (r1, w)
            if (REC) { R->rb[mr] = enc(u, p1(j)); R->Rx[mr + 1] = w; }
            mr++;
            ex = m1(j);
        }
        cur = u;
    }
    atomicOr(m.status, GA_ERR_CONS_WALK);
    return -1;
}

__global__ void k_cons_count(MeshDev m, const int2 *cv, int nc, int *done, int *cnt, int *rsize)
{
    GRID_STRIDE(c, nc) {
        int K = 0;
        if (!done[c]) {
            K = cons_walk<false>(m, cv[c].x, cv[c].y, nullptr, 0);
            if (K <= 0) {
                done[c] = 1;   // present already, or an error (status set)
                K = 0;
            }
        }
        cnt[c] = K;
        rsize[c] = K ? cons_region(K) : 0;
        if (K) atomicAdd(&m.counters[C_CONS_PEND], 1);
    }
}

// walks again, recording the cavity, and claims its slots (larger key = smaller constraint id)
__global__ void k_cons_collect(MeshDev m, const int2 *cv, int nc, const int *cnt, const int *roff, int *work,
                               int op)
{
    GRID_STRIDE(c, nc) {
        int K = cnt[c];
        if (!K) continue;
        ConsRegion R(work + roff[c], K);
        R.hdr[0] = 0;
        if (cons_walk<true>(m, cv[c].x, cv[c].y, &R, K) != K) {
            atomicOr(m.status, GA_ERR_CONS_WALK);
            continue;
        }
        unsigned long long key = ((unsigned long long)op << 32) | (0xffffffffu - (unsigned)c);
        for (int i = 0; i < K; i++) atomicMax(&m.claim[R.slots[i]], key);
    }
}

// boundary edge of the cavity on side k of new triangle T: the old cavity side `side` had the
// outside neighbour `out` (-1 on the hull); k_relink repairs the outside end
GA_INLINE void cons_boundary(const MeshDev &m, int T, int k, int side, int out)
{
    set_link(m, T, k, mark_old(out));
    ((int *)(m.remap + enc_t(side)))[enc_j(side)] = enc(T, k);
}

// Triangulates the pseudo-polygon E(0), E(1..M), E(M + 1) lying left of E(0) -> E(M + 1), with
// E(i) = X[i] (or X[M + 1 - i] when rev); bs / bo: cavity side and outside neighbour of the
// boundary edge between E(i) and E(i + 1) at index i (M - i when rev).  New triangles take slots
// from slots[*s]; returns the triangle on the base edge E(0) E(M + 1) (its side 2).
// Run by one thread (width 1) or one wave (width 64).  In a wave every lane runs the same
// sequential control flow on the same values (the stack in stk is written with identical values
// by all lanes, and each lane reads its own writes); only the choice of the chain vertex is split
// across lanes, and only lane 0 writes the mesh.
__device__ int cons_fill(const MeshDev &m, const int *X, int M, bool rev, const int *bs, const int *bo,
                         const int *slots, int *s, int *stk, int lane, int width)
{
#define CE(i) (rev ? X[M + 1 - (i)] : X[(i)])
#define CB(i) (rev ? M - (i) : (i))
    int top = -1, sp = 0;
    stk[0] = 1; stk[1] = M; stk[2] = -1;
    sp = 1;
    while (sp > 0) {
        sp--;
        int lo = stk[3 * sp], hi = stk[3 * sp + 1], pe = stk[3 * sp + 2];
        int x = CE(lo - 1), y = CE(hi + 1);
        // the chain vertex whose circle through x and y holds no other chain vertex: the minimum
        // of the order "inside the circle of" (the circles through x and y on one side are
        // nested, and the tie-break makes the order strict).  Each lane scans a strided part,
        // a butterfly combines them, and every lane ends with the index a sequential scan finds.
        int ci = -1;
        for (int i = lo + lane; i <= hi; i += width)
            if (ci < 0 || incircle_dev(m, x, y, CE(ci), CE(i)) > 0) ci = i;
        if (width == 64)
            for (int d = 32; d > 0; d >>= 1) {
                int o = __shfl_xor(ci, d, 64);
                if (o >= 0 && (ci < 0 || incircle_dev(m, x, y, CE(ci), CE(o)) > 0)) ci = o;
            }
        int cv = CE(ci);
        int T = slots[(*s)++];
        if (lane == 0) {
            m.tv[T] = make_int4(x, y, cv, 0);
            if (orient_dev(m, m.pos[x], m.pos[y], m.pos[cv]) <= 0) atomicOr(m.status, GA_ERR_CONS_TRI);
            if (pe >= 0) {
                set_link(m, T, 2, pe);
                set_link(m, enc_t(pe), enc_j(pe), enc(T, 2));
            }
            // side 1: edge (cv, x); side 0: edge (y, cv)
            if (ci == lo) cons_boundary(m, T, 1, bs[CB(lo - 1)], bo[CB(lo - 1)]);
            if (ci == hi) cons_boundary(m, T, 0, bs[CB(hi)], bo[CB(hi)]);
            m.vt[x] = T;
            m.vt[y] = T;
            m.vt[cv] = T;
        }
        if (pe < 0) top = T;
        if (ci > lo) {
            stk[3 * sp] = lo; stk[3 * sp + 1] = ci - 1; stk[3 * sp + 2] = enc(T, 1);
            sp++;
        }
        if (ci < hi) {
            stk[3 * sp] = ci + 1; stk[3 * sp + 1] = hi; stk[3 * sp + 2] = enc(T, 0);
            sp++;
        }
    }
#undef CE
#undef CB
    return top;
}

// Cavities below CONS_WAVE_K triangles: one thread per constraint; larger ones: one wave per
// constraint (wave-uniform control flow throughout).  A slot belongs to at most one winning
// cavity, so the two kernels never touch the same slots.
#define CONS_WAVE_K 32

__device__ void cons_commit_one(const MeshDev &m, int c, int K, int *done, const int *roff, int *work,
                                int *modlist, int op, int lane, int width)
{
    ConsRegion R(work + roff[c], K);
    if (R.hdr[0] != K) return;   // collect failed (status set)
    unsigned long long key = ((unsigned long long)op << 32) | (0xffffffffu - (unsigned)c);
    bool lost = false;
    for (int i = lane; i < K; i += width) lost |= m.claim[R.slots[i]] != key;
    if (width == 64 ? __ballot(lost) != 0 : lost) return;
    int ml = R.hdr[1], mr = R.hdr[2];
    // outside neighbours of the boundary, read before any slot is rewritten (every lane writes
    // the whole list, so it reads back only its own writes)
    for (int i = 0; i <= ml; i++) R.ol[i] = ic(m.tn[enc_t(R.lb[i])], enc_j(R.lb[i]));
    for (int i = 0; i <= mr; i++) R.orr[i] = ic(m.tn[enc_t(R.rb[i])], enc_j(R.rb[i]));
    for (int i = lane; i < K; i += width) m.stamp[R.slots[i]] = op;
    int s = 0;
    int tl = cons_fill(m, R.Lx, ml, false, R.lb, R.ol, R.slots, &s, R.stk, lane, width);
    int tr = cons_fill(m, R.Rx, mr, true, R.rb, R.orr, R.slots, &s, R.stk, lane, width);
    int q = 0;
    if (lane == 0) {
        set_link(m, tl, 2, enc(tr, 2));   // the constraint edge (a, b)
        set_link(m, tr, 2, enc(tl, 2));
        q = atomicAdd(&m.counters[C_CONS_MOD], K);
        done[c] = 1;
    }
    if (width == 64) q = __shfl(q, 0, 64);
    for (int i = lane; i < K; i += width) modlist[q + i] = R.slots[i];
}

// (the bound: without it the compiler keeps to 128 registers, for 1,024 threads, and spills; 96 us per launch
// for 10,000 constraints at 100,000 points without, 58 with)
__global__ __launch_bounds__(256) void k_cons_commit_small(MeshDev m, int nc, int *done, const int *cnt,
                                                           const int *roff, int *work, int *modlist, int op)
{
    GRID_STRIDE(c, nc) {
        int K = cnt[c];
        if (K > 0 && K < CONS_WAVE_K) cons_commit_one(m, c, K, done, roff, work, modlist, op, 0, 1);
    }
}

__global__ __launch_bounds__(256) void k_cons_commit_wave(MeshDev m, int nc, int *done, const int *cnt,
                                                          const int *roff, int *work, int *modlist, int op)
{
    int lane = threadIdx.x & 63;
    int wave = (blockIdx.x * blockDim.x + threadIdx.x) >> 6, nw = (gridDim.x * blockDim.x) >> 6;
    for (int c = wave; c < nc; c += nw) {
        int K = cnt[c];
        if (K >= CONS_WAVE_K) cons_commit_one(m, c, K, done, roff, work, modlist, op, lane, 64);
    }
}

void launch_cons_setup(MeshDev &m, const int2 *cin, int nc, int *inv, int2 *cv, int *done,
                       unsigned long long *chash, int chmask, hipStream_t st)
{
    GA_LAUNCH(k_cons_inv, dim3(FIXED_GRID), dim3(256), 0, st, m, inv);
    GA_LAUNCH(k_cons_map, dim3(FIXED_GRID), dim3(256), 0, st, m, cin, nc, (const int *)inv, cv, done, chash, chmask);
    GA_LAUNCH(k_cons_vt, dim3(FIXED_GRID), dim3(256), 0, st, m);
}

void launch_cons_count(MeshDev &m, const int2 *cv, int nc, int *done, int *cnt, int *rsize, hipStream_t st)
{
    GA_LAUNCH(k_cons_count, dim3(FIXED_GRID), dim3(256), 0, st, m, cv, nc, done, cnt, rsize);
}

void launch_cons_insert(MeshDev &m, const int2 *cv, int nc, int *done, const int *cnt, const int *roff,
                        int *work, int *modlist, int op, hipStream_t st)
{
    GA_LAUNCH(k_cons_collect, dim3(FIXED_GRID), dim3(256), 0, st, m, cv, nc, cnt, roff, work, op);
    GA_LAUNCH(k_cons_commit_small, dim3(FIXED_GRID), dim3(256), 0, st, m, nc, done, cnt, roff, work, modlist, op);
    GA_LAUNCH(k_cons_commit_wave, dim3(FIXED_GRID), dim3(256), 0, st, m, nc, done, cnt, roff, work, modlist, op);
    GA_LAUNCH(k_relink, dim3(FIXED_GRID), dim3(256), 0, st, m, (const int *)modlist, C_CONS_MOD, op, -1);
}
