// pba.hip -- discrete Voronoi diagram on a T x T texture (gfx950).
//
// Replaces the reference's PBA path (Cuda/pba2DHost.cu:82-155, Cuda/pba2DKernel.h:48-477,
// Cuda/kernelVoronoi.h:48-191, Cuda/cudaVoronoi.cu:181-307) with a layout and kernels of
// its own:
//   * textures are x-major (pixel (x, y) at x*T + y), so a wave whose lanes are 64
//     consecutive rows reads and writes 256 contiguous bytes per column step;
//   * phase 1 (nearest site in each column) is one wave per column: a 64-bit ballot per
//     64-row chunk marks the sites, and the nearest site above/below each pixel comes from
//     bit scans over those masks held in LDS -- the site map is read once;
//   * phases 2 and 3 are one search of the column field outward from every pixel, in LDS
//     tiles; only pixels far from every site take a second kernel (see there).
// All distances are exact integers; every pixel receives a site at minimal Euclidean
// distance (ties go to the lower column, then the lower row).
//
// The island certificate replaces the reference's iterate-and-recolour loop
// (kernelIslandDetection, CPU colorIsland): a pixel must have a same-labelled neighbour
// one step toward its site (dx, dy or the diagonal).  Sites failing it are taken out of
// the site map and the diagram is repaired: their columns get new nearest sites, their pixels
// the nearest site that is left, so every label stays an exact nearest site.
#include "dev_common.h"
#include "kernels.h"
#include <algorithm>

#define PBA_EMPTY 0x7fffffff

__global__ void k_fill_i32(int *a, int v, size_t n)
{
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    size_t stride = (size_t)gridDim.x * blockDim.x;
    for (; i < n; i += stride) a[i] = v;
}

// Set of every vertex: real points by their poff range, frame vertices by their fbase range.
__global__ void k_vset(const SetDesc *__restrict__ sets, int nsets, int ntot, int V, int *__restrict__ vset)
{
    int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= V) return;
    int lo = 0, hi = nsets - 1;
    if (v < ntot) {
        while (lo < hi) {
            int mid = (lo + hi + 1) >> 1;
            if (sets[mid].poff <= v) lo = mid;
            else hi = mid - 1;
        }
    } else {
        while (lo < hi) {
            int mid = (lo + hi + 1) >> 1;
            if (sets[mid].fbase <= v) lo = mid;
            else hi = mid - 1;
        }
    }
    vset[v] = lo;
}

// pixel of a real point in its set's texture (clamped inside the margin)
GA_INLINE void point_pixel(const SetDesc &sd, double2 p, int *px_, int *py_)
{
    int margin = sd.margin;
    int px = (int)floor((p.x - sd.shx) * sd.inv) + margin;
    int py = (int)floor((p.y - sd.shy) * sd.inv) + margin;
    int T = 1 << sd.logT;
    *px_ = px < margin ? margin : (px > T - 1 - margin ? T - 1 - margin : px);
    *py_ = py < margin ? margin : (py > T - 1 - margin ? T - 1 - margin : py);
}

// Spatial order of the real points: a counting sort by 16 x 16-pixel cell, cells of a set in
// Morton order after the cells of the previous sets (SetDesc::coff).  The order inside a cell is
// arbitrary; rules that depend on point order (the pixel's site, insertion claims) use the
// input index.
GA_INLINE unsigned spread14(unsigned v)
{
    v &= 0x3fffu;
    v = (v | (v << 8)) & 0x00ff00ffu;
    v = (v | (v << 4)) & 0x0f0f0f0fu;
    v = (v | (v << 2)) & 0x33333333u;
    v = (v | (v << 1)) & 0x55555555u;
    return v;
}

// Bound by the atomics on the cells' counts: those of one block of 1,024 * PER points go through a table
// in LDS first, so that a cell takes one per block.  (One per point, and a second one in the scatter: 48
// + 78 us for 1M uniform points, 52 + 15 now; 137 + 97 for 250K in 8 clusters, whose cells are few and
// full, so that their atomics queue up on a few lines, 29 + under 10 now.)  PER is 4 from 128K points on, where that
// leaves blocks enough (250K in clusters: 69 us with 1, 29 with 4).  slot[i]: the point's place in its cell.
template <int PER>
__global__ __launch_bounds__(1024) void k_cell_count(const double2 *__restrict__ xy, BatchDev b, int *__restrict__ cell,
                                                     int *__restrict__ slot, int *__restrict__ ccount)
{
    constexpr int TAB = 2048 * PER;
    __shared__ int s_key[TAB], s_cnt[TAB];
    for (int k = threadIdx.x; k < TAB; k += 1024) {
        s_key[k] = -1;
        s_cnt[k] = 0;
    }
    __syncthreads();
    const int i0 = blockIdx.x * 1024 * PER + threadIdx.x;
    int h[PER], at[PER];
#pragma unroll
    for (int u = 0; u < PER; u++) {
        const int i = i0 + 1024 * u;
        h[u] = at[u] = 0;
        if (i >= b.ntot) continue;
        const SetDesc &sd = b.sets[b.vset[i]];
        int px, py;
        point_pixel(sd, xy[i], &px, &py);
        const int c = sd.coff + (int)((spread14((unsigned)px >> 4) << 1) | spread14((unsigned)py >> 4));
        cell[i] = c;
        for (h[u] = (int)(((unsigned)c * 0x9E3779B1u) % TAB);; h[u] = (h[u] + 1) % TAB) {
            const int k = atomicCAS(&s_key[h[u]], -1, c);
            if (k == -1 || k == c) break;
        }
        at[u] = atomicAdd(&s_cnt[h[u]], 1);
    }
    __syncthreads();
    for (int k = threadIdx.x; k < TAB; k += 1024)
        if (s_cnt[k]) s_cnt[k] = atomicAdd(&ccount[s_key[k]], s_cnt[k]);
    __syncthreads();
#pragma unroll
    for (int u = 0; u < PER; u++) {
        const int i = i0 + 1024 * u;
        if (i < b.ntot) slot[i] = s_cnt[h[u]] + at[u];
    }
}

// first = exclusive prefix of the cell counts; perm[new index] = input index
__global__ void k_cell_scatter(const int *__restrict__ cell, const int *__restrict__ slot, int n,
                               const int *__restrict__ first, int *__restrict__ perm)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) perm[first[cell[i]] + slot[i]] = i;
}

__global__ void k_gather_xy(const double2 *__restrict__ xy, const int *__restrict__ perm, int n,
                            double2 *__restrict__ out)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = xy[perm[i]];
}

// Map real points to pixels of their set's texture.  pix = (px << 16) | py; the point with the
// smallest input index (perm[i], or i without a renumbering) wins a pixel; k_splat_own then
// stores the winner's own index.  Input indices carry SPLAT_INPUT (indices stay below 2^28), so that a
// thread of k_splat_own never takes another's own index, stored while it runs, for its input index.
#define SPLAT_INPUT 0x40000000
__global__ void k_splat(const double2 *__restrict__ xy, BatchDev b, const int *__restrict__ perm,
                        int *__restrict__ smap, int *__restrict__ pix)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= b.ntot) return;
    const SetDesc &sd = b.sets[b.vset[i]];
    int px, py;
    point_pixel(sd, xy[i], &px, &py);
    pix[i] = (px << 16) | py;
    atomicMin(&smap[sd.toff + ((size_t)px << sd.logT) + py], perm ? perm[i] | SPLAT_INPUT : i);
}

// The winners' own indices, and the frame sites (global ids ntot .. V-1) at their border pixels (fpix: packed
// local pixels).
__global__ void k_splat_own(BatchDev b, const int *__restrict__ perm, const int *__restrict__ fpix,
                            int *__restrict__ pix, int *__restrict__ smap)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= b.V || (i < b.ntot && !perm)) return;
    const SetDesc &sd = b.sets[b.vset[i]];
    const int pp = i < b.ntot ? pix[i] : fpix[i - b.ntot];
    int *cellp = &smap[sd.toff + ((size_t)(pp >> 16) << sd.logT) + (pp & 0xffff)];
    if (i >= b.ntot) {
        pix[i] = pp;
        *cellp = i;
    } else if (*cellp == (perm[i] | SPLAT_INPUT)) {
        *cellp = i;    // one winner per pixel: no other thread writes here
    }
}

// ---- phase 1: nearest site per column --------------------------------------------------
// One column, one wave (every wave of the block calls it): g[y] = row of the nearest site of the
// column (ties to the lower row), -1 for an empty column.  masks, prv, nxt: 256 LDS entries of the
// wave.
GA_INLINE void pba_column(const int *__restrict__ col, short *__restrict__ gc, int nch, int lane,
                          unsigned long long *masks, short *prv, short *nxt)
{
    for (int c = 0; c < nch; c++) {
        int v = col[(c << 6) + lane];
        unsigned long long m = __ballot(v != PBA_EMPTY);
        if (lane == 0) masks[c] = m;
    }
    __syncthreads();
    // previous / next nonempty chunk, 64 chunks per ballot group
    int carry_prev = -1;
    for (int gbase = 0; gbase < nch; gbase += 64) {
        int c = gbase + lane;
        bool nz = c < nch && masks[c] != 0ull;
        unsigned long long b = __ballot(nz);
        unsigned long long below = lane ? (b & ((1ull << lane) - 1ull)) : 0ull;
        int pv = below ? gbase + 63 - __clzll(below) : carry_prev;
        if (c < nch) prv[c] = (short)pv;
        if (b) carry_prev = gbase + 63 - __clzll(b);
    }
    int carry_next = nch;
    for (int gbase = ((nch - 1) >> 6) << 6; gbase >= 0; gbase -= 64) {
        int c = gbase + lane;
        bool nz = c < nch && masks[c] != 0ull;
        unsigned long long b = __ballot(nz);
        unsigned long long above = (lane == 63) ? 0ull : (b & (~0ull << (lane + 1)));
        int nx = above ? gbase + __ffsll((long long)above) - 1 : carry_next;
        if (c < nch) nxt[c] = (short)nx;
        if (b) carry_next = gbase + __ffsll((long long)b) - 1;
    }
    __syncthreads();
    for (int c = 0; c < nch; c++) {
        unsigned long long m = masks[c];
        int y = (c << 6) + lane;
        unsigned long long mb = (lane == 63) ? m : (m & ((2ull << lane) - 1ull));
        int yb = -1, ya = -1;
        if (mb) yb = (c << 6) + 63 - __clzll(mb);
        else {
            int p = prv[c];
            if (p >= 0) yb = (p << 6) + 63 - __clzll(masks[p]);
        }
        unsigned long long ma = m & (~0ull << lane);
        if (ma) ya = (c << 6) + __ffsll((long long)ma) - 1;
        else {
            int q = nxt[c];
            if (q < nch) ya = (q << 6) + __ffsll((long long)masks[q]) - 1;
        }
        int r;
        if (yb < 0) r = ya;
        else if (ya < 0) r = yb;
        else r = (y - yb <= ya - y) ? yb : ya;
        gc[y] = (short)r;
    }
}

// block = 256 (4 waves, one column each)
__global__ __launch_bounds__(256) void k_pba_cols(const int *__restrict__ smap_all,
                                                  short *__restrict__ g_all, BatchDev bd)
{
    __shared__ unsigned long long masks[4][256];
    __shared__ short prv[4][256], nxt[4][256];
    const int *bm = bd.bmap(BM_COLS);
    int set = set_of(bm, bd.nsets, blockIdx.x);
    const SetDesc &sd = bd.sets[set];
    const int wave = threadIdx.x >> 6;
    const size_t off = sd.toff + ((size_t)((blockIdx.x - bm[set]) * 4 + wave) << sd.logT);
    pba_column(smap_all + off, g_all + off, (1 << sd.logT) >> 6, threadIdx.x & 63, masks[wave], prv[wave], nxt[wave]);
}

// ---- phases 2 and 3: nearest site per pixel ---------------------------------------------
// The nearest site of pixel (x, y) lies in column x +- k with k * k no larger than the best squared
// distance so far, so the columns are searched outward from x.  With 16 pixels and more per point
// that ends after a few columns: k_pba_label holds the squared row distances of a 64 x 64-pixel tile
// and 16 columns on either side in LDS and finds nearly every label of an evenly filled texture
// there, in one pass.  Pixels that are further from every site (the empty space between
// clusters) are left to the far kernels, which skip 16 and 64 columns at a time by their smallest
// row distance.  k_pba_label is bound by its LDS reads, the far kernels by their instructions; a
// stack of each row's envelope (a band of 64 columns per thread, then pairwise merges, compaction
// and a colouring pass) is one serial chain per row and took, at T = 4096 (1M uniform points), 284 us
// against 47; at T = 8192 (4M) 1,344 against 332; at T = 2048 with 8 clusters (mostly far pixels)
// 259 against 99.
#define LAB_R 16                     // columns searched on either side in the tile
#define LAB_W (64 + 2 * LAB_R)
#define LAB_EMPTY 0x3fffffff         // above every squared distance
#define LAB_FAR (-2)                 // label of a pixel left to the far kernels
#define FAR_ROWS_T 4096              // largest texture side of k_pba_far_rows
#define FAR_EMPTY 12000              // its row offset of an empty column: the square is above FAR_NONE, and 16 times
                                     // a squared distance with it is below 2^32
#define FAR_NONE 100000000           // above the squared distances of textures up to FAR_ROWS_T

GA_INLINE int site_at(const int *smap, const short *g, int logT, int x, int y)
{
    const size_t c = (size_t)x << logT;
    return smap[c + g[c + y]];
}

// One 64 x 64-pixel tile per block.  A lane takes two neighbouring rows of a column: both keys of a
// candidate are one LDS word, 64 * (squared distance) + 16 + (its column - x), so that the smaller key is the
// nearer site and, in ties, the lower column, and two rows take a packed add and a packed minimum
// (with a separate distance and column per row the compares and selects bound it: 1,510 us in a
// batch of 1,024 sets, 268M pixels, against 954).  far[4 * tile + k] tells whether pixels of columns 16 k ..
// 16 k + 15 are left, setfar[set] whether any of the set's are (both zero on entry).  16 waves
// when there are fewer than 1,024 tiles (T = 512: 64 tiles, 23 us with 4 waves, 10 with 16), else 4, whose
// longer runs of columns share more of the site reads.
typedef unsigned short us2 __attribute__((ext_vector_type(2)));

template <int W>
__global__ __launch_bounds__(64 * W) void k_pba_label(const short *__restrict__ g_all, const int *__restrict__ smap_all,
                                                      int *__restrict__ vor_all, int *__restrict__ far,
                                                      int *__restrict__ setfar, BatchDev bd)
{
    __shared__ int4 s_q[LAB_W * 8];
    us2 *s_d = (us2 *)s_q;   // [LAB_W][32] row pairs: 64 * dy^2, 0x7fff above LAB_R and in empty columns
    const int *bm = bd.bmap(BM_LABEL);
    const int set = set_of(bm, bd.nsets, blockIdx.x);
    const SetDesc &sd = bd.sets[set];
    const int logT = sd.logT, T = 1 << logT, nb = T >> 6;
    const int lb = blockIdx.x - bm[set], x0 = (lb / nb) * 64, y0 = (lb % nb) * 64;
    const short *g = g_all + sd.toff;
    const int *smap = smap_all + sd.toff;
    int *vor = vor_all + sd.toff;
    // 8 rows per thread and step: 16 bytes of one column
    for (int q = threadIdx.x; q < LAB_W * 8; q += 64 * W) {
        const int c = q >> 3, r = (q & 7) * 8, x = x0 - LAB_R + c;
        short v[8];
        unsigned short o[8];
        int4 t = {-1, -1, -1, -1};
        if (x >= 0 && x < T) t = *(const int4 *)(g + ((size_t)x << logT) + y0 + r);
        __builtin_memcpy(v, &t, 16);
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const int dy = abs(v[i] - (y0 + r + i));
            o[i] = v[i] >= 0 && dy <= LAB_R ? (unsigned short)(64 * dy * dy) : (unsigned short)0x7fff;
        }
        __builtin_memcpy(&t, o, 16);
        s_q[q] = t;
    }
    __syncthreads();
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, y = y0 + 2 * (lane & 31);
    int pb0 = -1, pb1 = -1, id0 = 0, id1 = 0;    // the columns and sites of the pixels before
    bool left = false;
    for (int i = 0; i < 32 / W; i++) {
        const int xi = (64 / W) * w + (32 / W) * (lane >> 5) + i;
        const us2 *p = s_d + (LAB_R + xi) * 32 + (lane & 31);
        us2 best = p[0] + (unsigned short)16;
#pragma unroll
        for (int k0 = 1; k0 <= LAB_R; k0 += 4) {
            if (!__any(max(best.x, best.y) >= 64 * k0 * k0)) break;
#pragma unroll
            for (int k = k0; k < k0 + 4; k++) {
                best = __builtin_elementwise_min(best, p[-32 * k] + (unsigned short)(64 * k * k + 16 - k));
                best = __builtin_elementwise_min(best, p[32 * k] + (unsigned short)(64 * k * k + 16 + k));
            }
        }
        const bool d0 = best.x < 64 * (LAB_R + 1) * (LAB_R + 1), d1 = best.y < 64 * (LAB_R + 1) * (LAB_R + 1);
        const int b0 = x0 + xi - 16 + (best.x & 63), b1 = x0 + xi - 16 + (best.y & 63);
        if (d0 && b0 != pb0) id0 = site_at(smap, g, logT, pb0 = b0, y);
        if (d1 && b1 != pb1) id1 = site_at(smap, g, logT, pb1 = b1, y + 1);
        *(int2 *)(vor + ((size_t)(x0 + xi) << logT) + y) = make_int2(d0 ? id0 : LAB_FAR, d1 ? id1 : LAB_FAR);
        left |= !(d0 && d1);
    }
    if (__any(left) && lane == 0) {
        far[4 * (size_t)blockIdx.x + (64 / W) * w / 16] = 1;
        setfar[set] = 1;
    }
}

// smallest row distance of 16 consecutive columns in every row (0x7fff: no site in them); only for
// sets with far pixels
__global__ __launch_bounds__(256) void k_pba_blockmin(const short *__restrict__ g_all, short *__restrict__ hmin_all,
                                                      const int *__restrict__ setfar, BatchDev bd)
{
    const int *bm = bd.bmap(BM_LABEL);
    const int set = set_of(bm, bd.nsets, blockIdx.x);
    const SetDesc &sd = bd.sets[set];
    const int logT = sd.logT, T = 1 << logT, nb = T >> 6;
    if (!setfar[set] || T <= FAR_ROWS_T) return;
    const int lb = blockIdx.x - bm[set], xb = (lb / nb) * 4 + (threadIdx.x >> 6), y = (lb % nb) * 64 + (threadIdx.x & 63);
    const short *g = g_all + sd.toff;
    int mn = 0x7fff;
#pragma unroll
    for (int i = 0; i < 16; i++) {
        const int v = g[((size_t)(16 * xb + i) << logT) + y];
        if (v >= 0) mn = min(mn, abs(v - y));
    }
    hmin_all[(sd.toff >> 4) + ((size_t)xb << logT) + y] = (short)mn;
}

// The far pixels of textures up to FAR_ROWS_T: one block holds the whole column field of up to 16 rows in
// LDS (8 at T = 2048, 4 at 4096; fewer where that leaves less than two blocks per CU: a search is a
// few thousand cycles of one wave, and 16 rows at T = 512 are 32 blocks: 68 us against 23 with 2).
// Lanes are rows times 4 to 32 neighbouring columns (a group of columns); a wave takes up to 16
// groups.  The nearest column of a row does not decrease from pixel to pixel (for columns i < j the
// difference of the squared distances grows with x), so between two known pixels only the columns
// between theirs can win: each wave's first group comes first, then the middles of ever shorter
// intervals, and in the wide cells of empty space both ends mostly have the same site and nothing
// is left to search.  A search goes outward from x and is ruled out by the smallest row distance of
// 64 columns at a time, then of 16.
// Without the LDS copy every step of a search is a dependent read of L2: k_pba_far takes 186 us at
// T = 512 (12,007 points in 8 clusters) and 278 us at T = 2048 (250,001), this 15 and 81 us.
__global__ __launch_bounds__(1024) void k_pba_far_rows(const short *__restrict__ g_all, const int *__restrict__ smap_all,
                                                       const int *__restrict__ pix, int *__restrict__ vor_all,
                                                       const int *__restrict__ far_all,
                                                       const int *__restrict__ setfar, BatchDev bd)
{
    // [T / 4][RB][4] row offset of the column's site (FAR_EMPTY: none); [T][RB] nearest column of the waves'
    // pixels (-1: not known yet); the smallest magnitude of an offset in 16 columns [T / 16][RB], in 64
    extern __shared__ int4 s_far4[];
    short *s_dy = (short *)s_far4;
    const int *bm = bd.bmap(BM_ROWS);
    const int set = set_of(bm, bd.nsets, blockIdx.x);
    if (!setfar[set]) return;
    const SetDesc &sd = bd.sets[set];
    const int logT = sd.logT, T = 1 << logT, nb = T >> 6, RB = pba_far_rows(logT, bd.far_rows), lr = __ffs(RB) - 1;
    const int y0 = (blockIdx.x - bm[set]) << lr, tid = threadIdx.x;
    // parts of 16 columns with far pixels in the tiles of these rows
    const int *far = far_all + 4 * (size_t)bd.bmap(BM_LABEL)[set];
    int any = 0;
    for (int p = tid; p < (T >> 4); p += 1024) any |= far[4 * ((p >> 2) * nb + (y0 >> 6)) + (p & 3)];
    if (!__syncthreads_or(any)) return;
    const short *g = g_all + sd.toff;
    short *s_mn = s_dy + ((size_t)T << (lr + 1)), *s_m4 = s_mn + ((size_t)(T >> 4) << lr);
    auto at = [&](int c, int row) { return ((((c >> 2) << lr) + row) << 2) + (c & 3); };
    // (four reads in flight per thread in this and the next loop)
    for (int q0 = tid; q0 < (T << lr); q0 += 4096) {
        short v[4];
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int q = min(q0 + 1024 * u, (T << lr) - 1);
            v[u] = g[((size_t)(q >> lr) << logT) + y0 + (q & (RB - 1))];
        }
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int q = q0 + 1024 * u, row = q & (RB - 1);
            if (q < (T << lr)) s_dy[at(q >> lr, row)] = v[u] < 0 ? (short)FAR_EMPTY : (short)(v[u] - (y0 + row));
        }
    }
    const int *smap = smap_all + sd.toff;
    int *vor = vor_all + sd.toff;
    const int lane = tid & 63, w = tid >> 6, r = lane & (RB - 1), y = y0 + r;
    const int step = 64 >> lr, nG = (T >> 4) / step;   // columns of a group, groups of a wave
    const int xw = w * (T >> 4) + (lane >> lr);        // the lane's column in group 0
    short *s_wave = s_dy + ((size_t)T << lr) + (size_t)w * nG * 64, *s_col = s_wave + lane;   // group k at [64 k]
    unsigned open = 0;   // groups whose pixel is far
    for (int k0 = 0; k0 < nG; k0 += 4) {
        int v[4], sp[4];
#pragma unroll
        for (int u = 0; u < 4; u++) v[u] = vor[((size_t)(xw + min(k0 + u, nG - 1) * step) << logT) + y];
#pragma unroll
        for (int u = 0; u < 4; u++) sp[u] = v[u] < 0 ? -1 : pix[v[u]];
#pragma unroll
        for (int u = 0; u < 4; u++)
            if (k0 + u < nG) {
                s_col[64 * (k0 + u)] = (short)(sp[u] >> 16);
                open |= (unsigned)(v[u] == LAB_FAR) << (k0 + u);
            }
    }
    __syncthreads();
    for (int q = tid; q < ((T >> 4) << lr); q += 1024) {
        int mn = FAR_EMPTY;
        for (int u = 0; u < 16; u++) mn = min(mn, abs((int)s_dy[at(16 * (q >> lr) + u, q & (RB - 1))]));
        s_mn[q] = (short)mn;
    }
    __syncthreads();
    for (int q = tid; q < ((T >> 6) << lr); q += 1024) {
        const int c = ((q >> lr) << (lr + 2)) + (q & (RB - 1));
        s_m4[q] = min(min(s_mn[c], s_mn[c + RB]), min(s_mn[c + 2 * RB], s_mn[c + 3 * RB]));
    }
    __syncthreads();
    // the nearest column of the pixels of group k among [lo, hi] (lanes with act; lo, hi: nearest
    // columns of known pixels of the row on either side, or the outermost columns)
    auto search = [&](int k, int lo, int hi, bool act) {
        const int x = xw + k * step, X = (w * (T >> 4) + k * step) >> 6;   // (a group lies in 64 columns)
        int best = -1, bx = -1;
        if (act) {
            best = FAR_NONE;
            const int vl = s_dy[at(lo, r)], vh = s_dy[at(hi, r)];
            const int el = __mul24(x - lo, x - lo) + __mul24(vl, vl), eh = __mul24(x - hi, x - hi) + __mul24(vh, vh);
            if (el < best) { best = el; bx = lo; }
            if (eh < best) { best = eh; bx = hi; }
        }
        // 64 columns that can hold a nearer site for some lane; 16 * (squared distance) + column as one
        // key: the smallest is the nearest of 16 columns, in ties the lower
        auto visit = [&](int B) {
            for (int b = 4 * B; b < 4 * B + 4; b++) {
                const int h = s_mn[(b << lr) + r], d = max(max(16 * b - x, x - (16 * b + 15)), 0);
                if (!__any(16 * b + 15 >= lo && 16 * b <= hi && __mul24(d, d) + __mul24(h, h) <= best)) continue;
                const int2 *p = (const int2 *)s_dy + ((4 * b) << lr) + r;
                const int a = x - 16 * b;
                int dx2 = __mul24(a, a);
                unsigned key = ~0u;
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const int2 t = p[q << lr];
                    const short v[4] = {(short)t.x, (short)(t.x >> 16), (short)t.y, (short)(t.y >> 16)};
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const int u = 4 * q + e;
                        key = min(key, ((unsigned)(v[e] * v[e] + dx2) << 4) + u);
                        dx2 += 2 * u + 1 - 2 * a;
                    }
                }
                const int dd = (int)(key >> 4), cx = 16 * b + (int)(key & 15);
                if (dd < best || (dd == best && cx < bx)) { best = dd; bx = cx; }
            }
        };
        if (__any(act && 64 * X + 63 >= lo && 64 * X <= hi)) visit(X);
        for (int j = 1; j < nb; j++) {
            const int bl = X - j, br = X + j, dl = x - (64 * bl + 63), dr = 64 * br - x;
            const bool inl = bl >= 0 && __mul24(dl, dl) <= best && 64 * bl + 63 >= lo;
            const bool inr = br < nb && __mul24(dr, dr) <= best && 64 * br <= hi;
            if (!__any(inl || inr)) break;
            const int hl = inl && 64 * bl <= hi ? s_m4[(bl << lr) + r] : FAR_EMPTY;
            const int hr = inr && 64 * br + 63 >= lo ? s_m4[(br << lr) + r] : FAR_EMPTY;
            if (__any(__mul24(dl, dl) + __mul24(hl, hl) <= best)) visit(bl);
            if (__any(__mul24(dr, dr) + __mul24(hr, hr) <= best)) visit(br);
        }
        if (act) s_col[64 * k] = (short)bx;
    };
    {
        const bool act = s_col[0] < 0;
        if (__any(act)) search(0, 0, T - 1, act);
    }
    __syncthreads();
    if (!__any(open)) return;
    const int end = w < 15 ? s_wave[nG * 64 + r] : T - 1;   // nearest column of the next wave's first pixel
    for (int s = nG >> 1; s; s >>= 1)
        for (int k = s; k < nG; k += 2 * s) {
            const int lo = s_col[64 * (k - s)], hi = k + s < nG ? s_col[64 * (k + s)] : end;
            const bool mine = s_col[64 * k] < 0;
            if (mine && lo == hi) s_col[64 * k] = (short)lo;
            const bool act = mine && lo != hi;
            if (__any(act)) search(k, lo, hi, act);
        }
#pragma unroll 4
    for (int k = 0; k < nG; k++) {
        const int c = s_col[64 * k];
        if ((open >> k) & 1)
            vor[((size_t)(xw + k * step) << logT) + y] = smap[((size_t)c << logT) + y + s_dy[at(c, r)]];
    }
}

// The far pixels of larger textures, by tiles (64 x 64 pixels per block, lanes are rows).  The nearest
// column of a row does not decrease from pixel to pixel (for columns i < j the difference of the squared distances
// grows with x), so between two known pixels only the columns between theirs can win.  The two
// outer columns of the tile are searched in full, then the middles of ever shorter intervals; in
// the wide empty regions both ends mostly have the same site and nothing is left to search.  A
// search goes outward from x by blocks of 16 columns, into those whose smallest row distance (hmin)
// can beat the best so far.  One wave per pixel column in sequence, from the pixel before, took
// 443 us at T = 2048 with 8 clusters, this 278 us.
__global__ __launch_bounds__(256) void k_pba_far(const short *__restrict__ g_all, const short *__restrict__ hmin_all,
                                                 const int *__restrict__ smap_all, const int *__restrict__ pix,
                                                 int *__restrict__ vor_all, const int *__restrict__ far, BatchDev bd)
{
    __shared__ short s_col[64][64];   // nearest column of pixel (x, y), -1: not known yet
    __shared__ unsigned char s_far[64][64];
    const int4 parts = *(const int4 *)(far + 4 * (size_t)blockIdx.x);
    if (!(parts.x | parts.y | parts.z | parts.w)) return;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int *bm = bd.bmap(BM_LABEL);
    const int set = set_of(bm, bd.nsets, blockIdx.x);
    const SetDesc &sd = bd.sets[set];
    const int logT = sd.logT, T = 1 << logT, nb = T >> 6, nblk = T >> 4;
    if (T <= FAR_ROWS_T) return;
    const int lb = blockIdx.x - bm[set], x0 = (lb / nb) * 64, y = (lb % nb) * 64 + lane;
    const short *g = g_all + sd.toff + y, *hmin = hmin_all + (sd.toff >> 4) + y;
    const int *smap = smap_all + sd.toff;
    int *vor = vor_all + sd.toff + y;
    for (int i = w; i < 64; i += 4) {
        const int v = vor[(size_t)(x0 + i) << logT];
        s_far[i][lane] = v == LAB_FAR;
        s_col[i][lane] = v == LAB_FAR ? (short)-1 : (short)(pix[v] >> 16);
    }
    __syncthreads();
    // the nearest column of pixel x0 + i among [lo, hi] (lanes with act)
    auto search = [&](int i, int lo, int hi, bool act) {
        const int x = x0 + i;
        int best = -1, bx = -1;
        if (act) {
            best = LAB_EMPTY;
            const int vl = g[(size_t)lo << logT], vh = g[(size_t)hi << logT];   // the ends' own sites bound it
            if (vl >= 0) { best = (x - lo) * (x - lo) + (vl - y) * (vl - y); bx = lo; }
            if (vh >= 0) {
                const int d = (x - hi) * (x - hi) + (vh - y) * (vh - y);
                if (d < best) { best = d; bx = hi; }
            }
        }
        const int b0 = lo >> 4, b1 = hi >> 4, xb = x >> 4;
        auto look = [&](int b) {
#pragma unroll
            for (int u = 0; u < 16; u++) {
                const int cx = 16 * b + u, v = g[(size_t)cx << logT];
                const int d = (x - cx) * (x - cx) + (v - y) * (v - y);
                if (v >= 0 && (d < best || (d == best && cx < bx))) { best = d; bx = cx; }
            }
        };
        if (__any(act && xb >= b0 && xb <= b1)) look(xb);
        for (int j = 1; j < nblk; j += 4) {
            int hl[4], hr[4];
            bool more = false;
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const int bl = xb - j - u, br = xb + j + u, dl = x - (16 * bl + 15), dr = 16 * br - x;
                const bool inl = dl * dl <= best && bl >= 0, inr = dr * dr <= best && br < nblk;
                more |= (inl && bl >= b0) || (inr && br <= b1);
                hl[u] = inl && bl >= b0 && bl <= b1 ? hmin[(size_t)bl << logT] : 0x7fff;
                hr[u] = inr && br <= b1 && br >= b0 ? hmin[(size_t)br << logT] : 0x7fff;
            }
            if (!__any(more)) break;
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const int bl = xb - j - u, br = xb + j + u, dl = x - (16 * bl + 15), dr = 16 * br - x;
                if (__any(hl[u] != 0x7fff && dl * dl + hl[u] * hl[u] <= best)) look(bl);
                if (__any(hr[u] != 0x7fff && dr * dr + hr[u] * hr[u] <= best)) look(br);
            }
        }
        if (act) s_col[i][lane] = (short)bx;
    };
    if (w < 2) {
        const int i = w ? 63 : 0;
        const bool act = s_col[i][lane] < 0;
        if (__any(act)) search(i, 0, T - 1, act);
    }
    for (int s = 32; s; s >>= 1) {
        __syncthreads();
        for (int i = s * (2 * w + 1); i < 63; i += 8 * s) {
            const int lo = s_col[i - s][lane], hi = s_col[min(i + s, 63)][lane];
            const bool open = s_col[i][lane] < 0;
            if (open && lo == hi) s_col[i][lane] = (short)lo;
            const bool act = open && lo != hi;
            if (__any(act)) search(i, lo, hi, act);
        }
    }
    __syncthreads();
    int pc = -1, pid = 0;
    for (int i = 16 * w; i < 16 * w + 16; i++) {
        if (!s_far[i][lane]) continue;
        const int c = s_col[i][lane];
        if (c != pc) {
            pid = smap[((size_t)c << logT) + g[(size_t)c << logT]];
            pc = c;
        }
        vor[(size_t)(x0 + i) << logT] = pid;
    }
}

// ---- island certificate ------------------------------------------------------------------
// bad[s]: 0, BAD_SITE (a pixel of s fails the certificate), BAD_REMOVED (taken out of the site map)
#define BAD_SITE 1
#define BAD_REMOVED 2
GA_INLINE void island_fail(int s, int *bad, int *flag)
{
    bad[s] = BAD_SITE;
    *flag = 1;
}

// Blocks of 1,024 pixels (a texture has T * T >= 4096 pixels, T >= 64), four consecutive rows per
// thread, so a wave reads whole lines of its own and its neighbour columns; XCD k takes one
// contiguous eighth of the blocks, whose neighbour columns are then in its own L2.  Bound by the
// reads of the diagram: 136 us at T = 8192 (2.0 TB/s); one pixel per thread, in launch order, took 226 us,
// and 1,640 us against 754 us on a batch of 1,024 textures (357M pixels).
GA_INLINE void island_block(const int *__restrict__ vor_all, const int *__restrict__ pix, const BatchDev &bd, int blk,
                            int *__restrict__ bad, int *__restrict__ flag)
{
    const int *bm = bd.bmap(BM_PIX);
    int set = set_of(bm, bd.nsets, blk);
    const SetDesc &sd = bd.sets[set];
    int logT = sd.logT;
    int T = 1 << logT;
    const int *vor = vor_all + sd.toff;
    size_t idx = (size_t)(blk - bm[set]) * 1024 + 4 * threadIdx.x;
    const int x = (int)(idx >> logT), y0 = (int)(idx & (T - 1));
    const int4 own = *(const int4 *)(vor + idx);
    const int lab[4] = {own.x, own.y, own.z, own.w};
    int sp[4], need = 0;   // need: 1 the left column, 2 the right one
#pragma unroll
    for (int j = 0; j < 4; j++) {
        sp[j] = lab[j] < 0 ? (x << 16) | (y0 + j) : (j && lab[j] == lab[j - 1] ? sp[j - 1] : pix[lab[j]]);
        const int sx = sp[j] >> 16;
        need |= sx < x ? 1 : (sx > x ? 2 : 0);
    }
    // (a site lies inside the texture, so the column one step toward it does too)
    int4 left = make_int4(-1, -1, -1, -1), right = left;
    if (need & 1) left = *(const int4 *)(vor + idx - T);
    if (need & 2) right = *(const int4 *)(vor + idx + T);
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int s = lab[j], sx = sp[j] >> 16, sy = sp[j] & 0xffff, y = y0 + j;
        const int dx = (sx > x) - (sx < x), dy = (sy > y) - (sy < y);
        if (dx == 0 && dy == 0) continue;
        const int lj = j == 0 ? left.x : (j == 1 ? left.y : (j == 2 ? left.z : left.w));
        const int rj = j == 0 ? right.x : (j == 1 ? right.y : (j == 2 ? right.z : right.w));
        bool ok = dx != 0 && (dx < 0 ? lj : rj) == s;
        if (!ok && dy != 0) {
            const int k = j + dy;
            const int v = k < 0 || k > 3 ? vor[idx + k] : (k == 0 ? own.x : (k == 1 ? own.y : (k == 2 ? own.z : own.w)));
            ok = v == s;
        }
        if (!ok && dx != 0 && dy != 0) ok = vor[idx + j + dy + ((long long)dx << logT)] == s;
        if (!ok) island_fail(s, bad, flag);
    }
}

__global__ __launch_bounds__(256) void k_islands(const int *__restrict__ vor_all, const int *__restrict__ pix,
                                                 BatchDev bd, int *__restrict__ bad, int *__restrict__ flag)
{
    const unsigned nb = gridDim.x, q8 = nb >> 3;   // the last nb % 8 blocks keep their numbers
    const unsigned blk = blockIdx.x < 8 * q8 ? (blockIdx.x & 7u) * q8 + (blockIdx.x >> 3) : blockIdx.x;
    island_block(vor_all, pix, bd, (int)blk, bad, flag);
}

// Takes the sites flagged by the certificate out of the site map, and lists them (count in *removed).
__global__ void k_remove_bad(int *__restrict__ bad, const int *__restrict__ pix, BatchDev bd,
                             int *__restrict__ smap, int *__restrict__ removed, int *__restrict__ rlist,
                             int *__restrict__ setbad)
{
    int s = blockIdx.x * blockDim.x + threadIdx.x;
    bool r = s < bd.ntot && bad[s] == BAD_SITE;
    const int k = wave_reserve(removed, r);
    if (!r) return;
    bad[s] = BAD_REMOVED;
    rlist[k] = s;
    const int set = bd.vset[s];
    setbad[set] = 1;
    const SetDesc &sd = bd.sets[set];
    int sp = pix[s];
    smap[sd.toff + ((size_t)(sp >> 16) << sd.logT) + (sp & 0xffff)] = PBA_EMPTY;
}

// phase 1 again for the columns of the removed sites [first, *removed) (one wave per block)
__global__ __launch_bounds__(64) void k_repair_cols(const int *__restrict__ rlist, int first,
                                                    const int *__restrict__ removed, const int *__restrict__ pix,
                                                    BatchDev bd, const int *__restrict__ smap_all,
                                                    short *__restrict__ g_all)
{
    __shared__ unsigned long long masks[256];
    __shared__ short prv[256], nxt[256];
    const int n = *removed;
    for (int k = first + blockIdx.x; k < n; k += gridDim.x) {
        const int s = rlist[k];
        const SetDesc &sd = bd.sets[bd.vset[s]];
        const size_t off = sd.toff + ((size_t)(pix[s] >> 16) << sd.logT);
        pba_column(smap_all + off, g_all + off, (1 << sd.logT) >> 6, threadIdx.x, masks, prv, nxt);
        __syncthreads();
    }
}

// The pixels of removed sites get the nearest site that is left, from the column field: columns at
// growing distance k on both sides while k * k can still win, with phase 3's ties (lower column).
// A wave holds 64 rows of one column, so its column reads are whole lines; four distances are in
// flight.  A repair takes 0.15 ms at T = 2048 and 0.3 ms at T = 8192, where a whole second diagram took
// 0.4 and 2.2 ms, and a batch of 1,024 sets (10-20% of them repaired, three times) 1.5 instead of 17 ms.
// Only these pixels need the certificate again (any other keeps its label, and the
// neighbour that certified it had the same one): the blocks of 1,024 pixels that hold some are listed.  Sets
// without a removed site return at once.
__global__ __launch_bounds__(256) void k_relabel(int *__restrict__ vor_all, const short *__restrict__ g_all,
                                                 const int *__restrict__ smap_all, const int *__restrict__ bad,
                                                 const int *__restrict__ setbad, BatchDev bd,
                                                 int *__restrict__ changed, int *__restrict__ nchanged)
{
    const int *bm = bd.bmap(BM_PIX);
    int set = set_of(bm, bd.nsets, blockIdx.x);
    if (!setbad[set]) return;
    const SetDesc &sd = bd.sets[set];
    const int logT = sd.logT, T = 1 << logT;
    int *vor = vor_all + sd.toff;
    const short *g = g_all + sd.toff;
    const int *smap = smap_all + sd.toff;
    bool any = false;
    for (int q = 0; q < 4; q++) {
        const size_t idx = (size_t)(blockIdx.x - bm[set]) * 1024 + q * 256 + threadIdx.x;
        const int s = vor[idx];
        const bool act = s >= 0 && bad[s] == BAD_REMOVED;
        if (!__any(act)) continue;
        any = any || act;
        const int x = (int)(idx >> logT), y = (int)(idx & (T - 1));
        long long best = act ? 0x7fffffffffffffffll : -1;
        int bx = -1, by = 0;
        for (int k = 0; k < T && __any((long long)k * k <= best); k += 4) {
            short gl[4], gr[4];
#pragma unroll
            for (int u = 0; u < 4; u++) {
                gl[u] = x - k - u >= 0 ? g[((size_t)(x - k - u) << logT) + y] : (short)-1;
                gr[u] = x + k + u < T ? g[((size_t)(x + k + u) << logT) + y] : (short)-1;
            }
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const long long kk = (long long)(k + u) * (k + u);
                if (gl[u] >= 0) {
                    const long long d = kk + (long long)(gl[u] - y) * (gl[u] - y);
                    if (d <= best) { best = d; bx = x - k - u; by = gl[u]; }
                }
                if (gr[u] >= 0) {
                    const long long d = kk + (long long)(gr[u] - y) * (gr[u] - y);
                    if (d < best) { best = d; bx = x + k + u; by = gr[u]; }
                }
            }
        }
        if (act) vor[idx] = bx < 0 ? -1 : smap[((size_t)bx << logT) + by];
    }
    if (__syncthreads_or(any) && threadIdx.x == 0) changed[atomicAdd(nchanged, 1)] = (int)blockIdx.x;
}

// the certificate of the listed blocks
__global__ __launch_bounds__(256) void k_recheck(const int *__restrict__ vor_all, const int *__restrict__ pix, BatchDev bd,
                                                 const int *__restrict__ changed, const int *__restrict__ nchanged,
                                                 int *__restrict__ bad, int *__restrict__ flag)
{
    const int n = *nchanged;
    for (int c = blockIdx.x; c < n; c += gridDim.x) island_block(vor_all, pix, bd, changed[c], bad, flag);
}

// ---- host-side launchers ---------------------------------------------------------------
void launch_fill_i32(int *a, int v, size_t n, hipStream_t st)
{
    int blocks = (int)((n + 255) / 256);
    if (blocks > 65536) blocks = 65536;
    if (blocks < 1) blocks = 1;
    GA_LAUNCH(k_fill_i32, dim3(blocks), dim3(256), 0, st, a, v, n);
}

void launch_vset(const BatchDev &b, int *vset, hipStream_t st)
{
    if (b.V > 0)
        GA_LAUNCH(k_vset, dim3((b.V + 255) / 256), dim3(256), 0, st, b.sets, b.nsets, b.ntot, b.V, vset);
}

// ccount (ncells + 1 entries) must be zero on entry
void launch_renumber(const double2 *xy, const BatchDev &b, int *cell, int *slot, int *ccount, int *first, int ncells,
                     void *scan_tmp, int *perm, double2 *xys, hipStream_t st)
{
    int n = b.ntot;
    if (n <= 0) return;
    if (n >= (1 << 17))
        GA_LAUNCH(k_cell_count<4>, dim3((n + 4095) / 4096), dim3(1024), 0, st, xy, b, cell, slot, ccount);
    else
        GA_LAUNCH(k_cell_count<1>, dim3((n + 1023) / 1024), dim3(1024), 0, st, xy, b, cell, slot, ccount);
    launch_exclusive_scan(ccount, first, (size_t)ncells + 1, scan_tmp, st);
    GA_LAUNCH(k_cell_scatter, dim3((n + 255) / 256), dim3(256), 0, st, (const int *)cell, (const int *)slot, n,
              (const int *)first, perm);
    GA_LAUNCH(k_gather_xy, dim3((n + 255) / 256), dim3(256), 0, st, xy, (const int *)perm, n, xys);
}

void launch_splat(const double2 *xy, const BatchDev &b, const int *perm, int *smap, int *pix, const int *fpix,
                  hipStream_t st)
{
    if (b.ntot > 0) GA_LAUNCH(k_splat, dim3((b.ntot + 255) / 256), dim3(256), 0, st, xy, b, perm, smap, pix);
    GA_LAUNCH(k_splat_own, dim3((b.V + 255) / 256), dim3(256), 0, st, b, perm, fpix, pix, smap);
}

void launch_pba(const PbaBuffers &p, const int *pix, const BatchDev &b, hipStream_t st)
{
    GA_LAUNCH(k_pba_cols, dim3(b.blocks[BM_COLS]), dim3(256), 0, st, p.smap, p.g, b);
    const int tiles = b.blocks[BM_LABEL];
    if (tiles < 1024)
        GA_LAUNCH(k_pba_label<16>, dim3(tiles), dim3(1024), 0, st, (const short *)p.g, (const int *)p.smap, p.vor, p.far,
                  p.setfar, b);
    else
        GA_LAUNCH(k_pba_label<4>, dim3(tiles), dim3(256), 0, st, (const short *)p.g, (const int *)p.smap, p.vor, p.far,
                  p.setfar, b);
    if (b.maxT > FAR_ROWS_T) {
        GA_LAUNCH(k_pba_blockmin, dim3(b.blocks[BM_LABEL]), dim3(256), 0, st, (const short *)p.g, p.hmin,
                  (const int *)p.setfar, b);
        GA_LAUNCH(k_pba_far, dim3(b.blocks[BM_LABEL]), dim3(256), 0, st, (const short *)p.g, (const short *)p.hmin,
                  (const int *)p.smap, pix, p.vor, (const int *)p.far, b);
    }
    if (b.blocks[BM_ROWS] > 0) {
        if (b.far_lds > 65536)
            (void)hipFuncSetAttribute((const void *)k_pba_far_rows, hipFuncAttributeMaxDynamicSharedMemorySize, b.far_lds);
        GA_LAUNCH(k_pba_far_rows, dim3(b.blocks[BM_ROWS]), dim3(1024), b.far_lds, st, (const short *)p.g, (const int *)p.smap, pix,
                  p.vor, (const int *)p.far, (const int *)p.setfar, b);
    }
}

void launch_islands(const int *vor, const int *pix, const BatchDev &b, int *bad, int *flag, hipStream_t st)
{
    GA_LAUNCH(k_islands, dim3(b.blocks[BM_PIX]), dim3(256), 0, st, vor, pix, b, bad, flag);
}

// removes the flagged sites (listed in rlist from position `first`, the number removed before) and
// repairs the diagram around them, then checks the blocks that changed (listed in changed); zeroes *flag and *nchanged
void launch_island_repair(const PbaBuffers &p, const BatchDev &b, int *bad, const int *pix, int *removed, int first,
                          int *rlist, int *changed, int *nchanged, int *flag, hipStream_t st)
{
    // (free after phase 3)
    int *setbad = p.setfar;
    if (b.ntot <= 0) return;
    IntFills f;
    f.add(setbad, (size_t)b.nsets, 0);
    f.add(nchanged, 1, 0);
    f.add(flag, 1, 0);
    launch_fill_multi(f, st);
    GA_LAUNCH(k_remove_bad, dim3((b.ntot + 255) / 256), dim3(256), 0, st, bad, pix, b, p.smap, removed, rlist, setbad);
    GA_LAUNCH(k_repair_cols, dim3(1024), dim3(64), 0, st, (const int *)rlist, first, (const int *)removed, pix, b,
              (const int *)p.smap, p.g);
    GA_LAUNCH(k_relabel, dim3(b.blocks[BM_PIX]), dim3(256), 0, st, p.vor, (const short *)p.g, (const int *)p.smap,
              (const int *)bad, (const int *)setbad, b, changed, nchanged);
    GA_LAUNCH(k_recheck, dim3(std::min(b.blocks[BM_PIX], 2048)), dim3(256), 0, st, (const int *)p.vor, pix, b,
              (const int *)changed, (const int *)nchanged, bad, flag);
}
