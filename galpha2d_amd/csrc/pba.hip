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
//   * phase 2 builds per-(row, band) stacks of proximate sites with lanes = rows, stored as
//     arrays (no pointer chasing), integer-exact dominance tests;
//   * phase 2b merges band stacks per row and compacts the envelope contiguously;
//   * phase 3 colours pixels with lanes = rows, binary-searching the start element of its
//     pixel band in the compacted envelope.
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

__global__ void k_cell_count(const double2 *__restrict__ xy, BatchDev b, int *__restrict__ cell,
                             int *__restrict__ ccount)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= b.ntot) return;
    const SetDesc &sd = b.sets[b.vset[i]];
    int px, py;
    point_pixel(sd, xy[i], &px, &py);
    int c = sd.coff + (int)((spread14((unsigned)px >> 4) << 1) | spread14((unsigned)py >> 4));
    cell[i] = c;
    atomicAdd(&ccount[c], 1);
}

// cursor = exclusive prefix of the cell counts; perm[new index] = input index
__global__ void k_cell_scatter(const int *__restrict__ cell, int n, int *__restrict__ cursor, int *__restrict__ perm)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) perm[atomicAdd(&cursor[cell[i]], 1)] = i;
}

__global__ void k_gather_xy(const double2 *__restrict__ xy, const int *__restrict__ perm, int n,
                            double2 *__restrict__ out)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = xy[perm[i]];
}

// Map real points to pixels of their set's texture.  pix = (px << 16) | py; the point with the
// smallest input index (perm[i], or i without a renumbering) wins a pixel; k_splat_own then
// stores the winner's own index.
__global__ void k_splat(const double2 *__restrict__ xy, BatchDev b, const int *__restrict__ perm,
                        int *__restrict__ smap, int *__restrict__ pix)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= b.ntot) return;
    const SetDesc &sd = b.sets[b.vset[i]];
    int px, py;
    point_pixel(sd, xy[i], &px, &py);
    pix[i] = (px << 16) | py;
    atomicMin(&smap[sd.toff + ((size_t)px << sd.logT) + py], perm ? perm[i] : i);
}

__global__ void k_splat_own(BatchDev b, const int *__restrict__ perm, const int *__restrict__ pix,
                            int *__restrict__ smap)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= b.ntot) return;
    const SetDesc &sd = b.sets[b.vset[i]];
    int pp = pix[i];
    int *cellp = &smap[sd.toff + ((size_t)(pp >> 16) << sd.logT) + (pp & 0xffff)];
    if (*cellp == perm[i]) *cellp = i;    // one winner per pixel: no other thread writes here
}

// Frame sites (global ids ntot .. V-1) at their border pixels (fpix: packed local pixels).
__global__ void k_splat_frame(const int *__restrict__ fpix, BatchDev b, int *__restrict__ smap,
                              int *__restrict__ pix)
{
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    int f = b.ntot + k;
    if (f >= b.V) return;
    const SetDesc &sd = b.sets[b.vset[f]];
    int pp = fpix[k];
    pix[f] = pp;
    smap[sd.toff + ((size_t)(pp >> 16) << sd.logT) + (pp & 0xffff)] = f;
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

// ---- phase 2: proximate-site stacks per (row, band) ------------------------------------
#define PBA_MAXB 64   // bands per texture row at most (m2, m3 <= 64)
GA_INLINE int pk(int x, int h) { return (x << 16) | (h & 0xffff); }
GA_INLINE int pk_x(int e) { return (int)((unsigned)e >> 16); }
GA_INLINE int pk_h(int e) { return (int)(short)(e & 0xffff); }

// b is dominated by a (left) and c (right): the a|b bisector is not left of the b|c one
GA_INLINE bool dominated(int a, int b, int c)
{
    long long xa = pk_x(a), ha = pk_h(a), xb = pk_x(b), hb = pk_h(b), xc = pk_x(c), hc = pk_h(c);
    long long fa = xa * xa + ha * ha, fb = xb * xb + hb * hb, fc = xc * xc + hc * hc;
    return (fb - fa) * (xc - xb) >= (fc - fb) * (xb - xa);
}

// grid (T/64, m2), block 64: lanes are rows.  Stack entries of band b live in
// S[(b*Wb + k) * T + y], k < hi[b*T + y]; lo[b*T + y] = 0 (the merge steps move both ends).
// The column reads of a band do not depend on the stack, so they are issued 8 at a time ahead
// of the dominance tests.
__global__ __launch_bounds__(64) void k_pba_stack(const short *__restrict__ g_all, int *__restrict__ S_all,
                                                  int *__restrict__ hi_all, int *__restrict__ lo_all, BatchDev bd)
{
    const int *bm = bd.bmap(BM_STACK);
    int set = set_of(bm, bd.nsets, blockIdx.x);
    const SetDesc &sd = bd.sets[set];
    int logT = sd.logT;
    int T = 1 << logT, nbx = T >> 6, Wb = T / sd.m2;
    int lb = blockIdx.x - bm[set];
    const short *g = g_all + sd.toff;
    int *S = S_all + sd.toff;
    size_t roff = (size_t)PBA_MAXB * sd.roff;
    int y = (lb % nbx) * 64 + threadIdx.x;
    int b = lb / nbx;
    int x0 = b * Wb;
    int top = 0, e0 = 0, e1 = 0;
    for (int xb = x0; xb < x0 + Wb; xb += 8) {
        short gv[8];
#pragma unroll
        for (int u = 0; u < 8; u++) gv[u] = xb + u < x0 + Wb ? g[((size_t)(xb + u) << logT) + y] : (short)-1;
#pragma unroll
        for (int u = 0; u < 8; u++) {
            int gy = gv[u];
            if (gy < 0) continue;
            int c = pk(xb + u, gy - y);
            while (top >= 2 && dominated(e0, e1, c)) {
                top--;
                e1 = e0;
                if (top >= 2) e0 = S[((size_t)(x0 + top - 2) << logT) + y];
            }
            S[((size_t)(x0 + top) << logT) + y] = c;
            top++;
            e0 = e1;
            e1 = c;
        }
    }
    hi_all[roff + (size_t)b * T + y] = top;
    lo_all[roff + (size_t)b * T + y] = 0;
}

// ---- phase 2b: merge band envelopes pairwise, then compact ------------------------------
// Step s merges, for every row, the envelope of bands [j*2^s, j*2^s + 2^(s-1)) with that of
// the next 2^(s-1) bands: the left chain's last element and the right chain's first are
// popped while the triple at the junction shows one of them dominated (the same exact test
// as the stacks).  A chain runs through the nonempty [lo, hi) ranges of its bands in order.
// The lower envelope of a row is unique, so the merge order does not change it.
// grid (T/64) * (m2/2) blocks of 64 (lanes are rows); blocks whose group does not exist at
// this step return.
__global__ __launch_bounds__(64) void k_pba_merge_step(const int *__restrict__ S_all, int *__restrict__ hi_all,
                                                       int *__restrict__ lo_all, BatchDev bd, int s)
{
    const int *bm = bd.bmap(BM_MERGE);
    int set = set_of(bm, bd.nsets, blockIdx.x);
    const SetDesc &sd = bd.sets[set];
    int logT = sd.logT;
    int T = 1 << logT, nbx = T >> 6, m2 = sd.m2, Wb = T / m2;
    int gsz = 1 << s, half = gsz >> 1;
    int lb = blockIdx.x - bm[set];
    int j = lb / nbx;
    if ((j + 1) * gsz > m2) return;
    const int *S = S_all + sd.toff;
    size_t roff = (size_t)PBA_MAXB * sd.roff;
    int y = (lb % nbx) * 64 + threadIdx.x;
    int *HI = hi_all + roff + y, *LO = lo_all + roff + y;   // band b at [b * T]
#define ELEM(B, I) S[((size_t)((B) * Wb + (I)) << logT) + y]
    int b0 = j * gsz, bmid = b0 + half, b1 = b0 + gsz;
    // L: last nonempty band of the left half; R: first nonempty band of the right half
    int L = bmid - 1;
    while (L >= b0 && HI[(size_t)L * T] <= LO[(size_t)L * T]) L--;
    int R = bmid;
    while (R < b1 && HI[(size_t)R * T] <= LO[(size_t)R * T]) R++;
    if (L < b0 || R >= b1) return;
    int Llo = LO[(size_t)L * T], Lhi = HI[(size_t)L * T];
    int Rlo = LO[(size_t)R * T], Rhi = HI[(size_t)R * T];
    for (;;) {
        int l1 = ELEM(L, Lhi - 1), r1 = ELEM(R, Rlo);
        // element before l1 on the left chain
        bool has0 = false;
        int l0 = 0;
        if (Lhi - 1 > Llo) { l0 = ELEM(L, Lhi - 2); has0 = true; }
        else {
            int P = L - 1;
            while (P >= b0 && HI[(size_t)P * T] <= LO[(size_t)P * T]) P--;
            if (P >= b0) { l0 = ELEM(P, HI[(size_t)P * T] - 1); has0 = true; }
        }
        if (has0 && dominated(l0, l1, r1)) {
            Lhi--;
            HI[(size_t)L * T] = Lhi;
            if (Lhi == Llo) {
                L--;
                while (L >= b0 && HI[(size_t)L * T] <= LO[(size_t)L * T]) L--;
                if (L < b0) break;
                Llo = LO[(size_t)L * T]; Lhi = HI[(size_t)L * T];
            }
            continue;
        }
        // element after r1 on the right chain
        bool has2 = false;
        int r2 = 0;
        if (Rlo + 1 < Rhi) { r2 = ELEM(R, Rlo + 1); has2 = true; }
        else {
            int Q = R + 1;
            while (Q < b1 && HI[(size_t)Q * T] <= LO[(size_t)Q * T]) Q++;
            if (Q < b1) { r2 = ELEM(Q, LO[(size_t)Q * T]); has2 = true; }
        }
        if (has2 && dominated(l1, r1, r2)) {
            Rlo++;
            LO[(size_t)R * T] = Rlo;
            if (Rlo == Rhi) {
                R++;
                while (R < b1 && HI[(size_t)R * T] <= LO[(size_t)R * T]) R++;
                if (R >= b1) break;
                Rlo = LO[(size_t)R * T]; Rhi = HI[(size_t)R * T];
            }
            continue;
        }
        break;
    }
#undef ELEM
}

// grid (T/64) * m2 blocks of 64 (lanes are rows): band b's [lo, hi) goes to the row's compacted
// envelope after the ranges of bands 0 .. b-1; the last band writes the envelope size
__global__ __launch_bounds__(64) void k_pba_compact(const int *__restrict__ S_all, const int *__restrict__ hi_all,
                                                    const int *__restrict__ lo_all, int *__restrict__ E_all,
                                                    int *__restrict__ ecnt_all, BatchDev bd)
{
    const int *bm = bd.bmap(BM_STACK);
    int set = set_of(bm, bd.nsets, blockIdx.x);
    const SetDesc &sd = bd.sets[set];
    int logT = sd.logT;
    int T = 1 << logT, nbx = T >> 6, m2 = sd.m2, Wb = T / m2;
    int lb = blockIdx.x - bm[set];
    int b = lb / nbx;
    int y = (lb % nbx) * 64 + threadIdx.x;
    size_t roff = (size_t)PBA_MAXB * sd.roff;
    const int *HI = hi_all + roff + y, *LO = lo_all + roff + y;
    int off = 0;
    for (int q = 0; q < b; q++) off += HI[(size_t)q * T] - LO[(size_t)q * T];
    int lo = LO[(size_t)b * T], hi = HI[(size_t)b * T];
    const int *S = S_all + sd.toff;
    int *E = E_all + sd.toff;
    for (int i = lo; i < hi; i++) E[((size_t)(off + i - lo) << logT) + y] = S[((size_t)(b * Wb + i) << logT) + y];
    if (b == m2 - 1) ecnt_all[sd.roff + y] = off + (hi > lo ? hi - lo : 0);
}

// ---- phase 3: colour ------------------------------------------------------------------
GA_INLINE long long fdist(int e, int i)
{
    long long dx = i - pk_x(e), h = pk_h(e);
    return dx * dx + h * h;
}

// grid (T/64, m3), block 64; vor[x*T + y] = site id
__global__ __launch_bounds__(64) void k_pba_color(const int *__restrict__ E_all, const int *__restrict__ ecnt_all,
                                                  const int *__restrict__ smap_all, int *__restrict__ vor_all,
                                                  BatchDev bd)
{
    const int *bm = bd.bmap(BM_COLOR);
    int set = set_of(bm, bd.nsets, blockIdx.x);
    const SetDesc &sd = bd.sets[set];
    int logT = sd.logT;
    int T = 1 << logT, nbx = T >> 6, Wp = T / sd.m3;
    int lb = blockIdx.x - bm[set];
    const int *E = E_all + sd.toff;
    const int *ecnt = ecnt_all + sd.roff;
    const int *smap = smap_all + sd.toff;
    int *vor = vor_all + sd.toff;
    int y = (lb % nbx) * 64 + threadIdx.x;
    int ps = (lb / nbx) * Wp, pe = ps + Wp;
    int n = ecnt[y];
    if (n <= 0) {
        for (int i = ps; i < pe; i++) vor[((size_t)i << logT) + y] = -1;
        return;
    }
#define EL(K) E[((size_t)(K) << logT) + y]
    int lo = 0, hi = n - 1;
    while (lo < hi) {
        int mid = (lo + hi) >> 1;
        if (fdist(EL(mid + 1), ps) < fdist(EL(mid), ps)) lo = mid + 1;
        else hi = mid;
    }
    int k = lo;
    int e = EL(k);
    int en = (k + 1 < n) ? EL(k + 1) : 0;
    int id = smap[((size_t)pk_x(e) << logT) + (y + pk_h(e))];
    for (int i = ps; i < pe; i++) {
        while (k + 1 < n && fdist(en, i) < fdist(e, i)) {
            k++;
            e = en;
            en = (k + 1 < n) ? EL(k + 1) : 0;
            id = smap[((size_t)pk_x(e) << logT) + (y + pk_h(e))];
        }
        vor[((size_t)i << logT) + y] = id;
    }
#undef EL
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
__global__ __launch_bounds__(256) void k_islands(const int *__restrict__ vor_all, const int *__restrict__ pix,
                                                 BatchDev bd, int *__restrict__ bad, int *__restrict__ flag)
{
    const unsigned nb = gridDim.x, q8 = nb >> 3;   // the last nb % 8 blocks keep their numbers
    const unsigned blk = blockIdx.x < 8 * q8 ? (blockIdx.x & 7u) * q8 + (blockIdx.x >> 3) : blockIdx.x;
    const int *bm = bd.bmap(BM_PIX);
    int set = set_of(bm, bd.nsets, (int)blk);
    const SetDesc &sd = bd.sets[set];
    int logT = sd.logT;
    int T = 1 << logT;
    const int *vor = vor_all + sd.toff;
    size_t idx = (size_t)((int)blk - bm[set]) * 1024 + 4 * threadIdx.x;
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
// neighbour that certified it had the same one): they are listed.  Blocks of 1,024 pixels; sets
// without a removed site return at once.
__global__ __launch_bounds__(256) void k_relabel(int *__restrict__ vor_all, const short *__restrict__ g_all,
                                                 const int *__restrict__ smap_all, const int *__restrict__ bad,
                                                 const int *__restrict__ setbad, BatchDev bd,
                                                 unsigned *__restrict__ changed, int *__restrict__ chset,
                                                 int *__restrict__ nchanged)
{
    const int *bm = bd.bmap(BM_PIX);
    int set = set_of(bm, bd.nsets, blockIdx.x);
    if (!setbad[set]) return;
    const SetDesc &sd = bd.sets[set];
    const int logT = sd.logT, T = 1 << logT;
    int *vor = vor_all + sd.toff;
    const short *g = g_all + sd.toff;
    const int *smap = smap_all + sd.toff;
    for (int q = 0; q < 4; q++) {
        const size_t idx = (size_t)(blockIdx.x - bm[set]) * 1024 + q * 256 + threadIdx.x;
        const int s = vor[idx];
        const bool act = s >= 0 && bad[s] == BAD_REMOVED;
        if (!__any(act)) continue;
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
        const int c = wave_reserve(nchanged, act);
        if (!act) continue;
        vor[idx] = bx < 0 ? -1 : smap[((size_t)bx << logT) + by];
        changed[c] = (unsigned)idx;
        chset[c] = set;
    }
}

// the certificate of the relabelled pixels (set and pixel of each)
__global__ void k_recheck(const int *__restrict__ vor_all, const int *__restrict__ pix, BatchDev bd,
                          const unsigned *__restrict__ changed, const int *__restrict__ chset,
                          const int *__restrict__ nchanged, int *__restrict__ bad, int *__restrict__ flag)
{
    const int n = *nchanged;
    for (int c = blockIdx.x * blockDim.x + threadIdx.x; c < n; c += gridDim.x * blockDim.x) {
        const SetDesc &sd = bd.sets[chset[c]];
        const size_t idx = changed[c];
        const int logT = sd.logT, T = 1 << logT;
        const int *vor = vor_all + sd.toff;
        const int s = vor[idx];
        if (s < 0) continue;
        const int x = (int)(idx >> logT), y = (int)(idx & (T - 1)), sp = pix[s], sx = sp >> 16, sy = sp & 0xffff;
        const int dx = (sx > x) - (sx < x), dy = (sy > y) - (sy < y);
        if (dx == 0 && dy == 0) continue;
        bool ok = dx != 0 && vor[idx + ((long long)dx << logT)] == s;
        if (!ok && dy != 0) ok = vor[idx + dy] == s;
        if (!ok && dx != 0 && dy != 0) ok = vor[idx + ((long long)dx << logT) + dy] == s;
        if (!ok) island_fail(s, bad, flag);
    }
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
void launch_renumber(const double2 *xy, const BatchDev &b, int *cell, int *ccount, int *cursor, int ncells,
                     void *scan_tmp, int *perm, double2 *xys, hipStream_t st)
{
    int n = b.ntot;
    if (n <= 0) return;
    GA_LAUNCH(k_cell_count, dim3((n + 255) / 256), dim3(256), 0, st, xy, b, cell, ccount);
    launch_exclusive_scan(ccount, cursor, (size_t)ncells + 1, scan_tmp, st);
    GA_LAUNCH(k_cell_scatter, dim3((n + 255) / 256), dim3(256), 0, st, (const int *)cell, n, cursor, perm);
    GA_LAUNCH(k_gather_xy, dim3((n + 255) / 256), dim3(256), 0, st, xy, (const int *)perm, n, xys);
}

void launch_splat(const double2 *xy, const BatchDev &b, const int *perm, int *smap, int *pix, const int *fpix,
                  hipStream_t st)
{
    if (b.ntot > 0) {
        GA_LAUNCH(k_splat, dim3((b.ntot + 255) / 256), dim3(256), 0, st, xy, b, perm, smap, pix);
        if (perm)
            GA_LAUNCH(k_splat_own, dim3((b.ntot + 255) / 256), dim3(256), 0, st, b, perm, (const int *)pix, smap);
    }
    int nf = b.V - b.ntot;
    if (nf > 0)
        GA_LAUNCH(k_splat_frame, dim3((nf + 255) / 256), dim3(256), 0, st, fpix, b, smap, pix);
}

void launch_pba(const PbaBuffers &p, const BatchDev &b, hipStream_t st)
{
    GA_LAUNCH(k_pba_cols, dim3(b.blocks[BM_COLS]), dim3(256), 0, st, p.smap, p.g, b);
    GA_LAUNCH(k_pba_stack, dim3(b.blocks[BM_STACK]), dim3(64), 0, st, p.g, p.S, p.cnt, p.lo, b);
    for (int s = 1; (1 << s) <= b.max_m2; s++)
        GA_LAUNCH(k_pba_merge_step, dim3(b.blocks[BM_MERGE]), dim3(64), 0, st, (const int *)p.S, p.cnt, p.lo, b, s);
    GA_LAUNCH(k_pba_compact, dim3(b.blocks[BM_STACK]), dim3(64), 0, st, (const int *)p.S, (const int *)p.cnt,
              (const int *)p.lo, p.E, p.ecnt, b);
    GA_LAUNCH(k_pba_color, dim3(b.blocks[BM_COLOR]), dim3(64), 0, st, p.E, p.ecnt, p.smap, p.vor, b);
}

void launch_islands(const int *vor, const int *pix, const BatchDev &b, int *bad, int *flag, hipStream_t st)
{
    GA_LAUNCH(k_islands, dim3(b.blocks[BM_PIX]), dim3(256), 0, st, vor, pix, b, bad, flag);
}

// removes the flagged sites (listed in rlist from position `first`, the number removed before) and
// repairs the diagram around them, then checks the pixels that changed; zeroes *flag and *nchanged
void launch_island_repair(const PbaBuffers &p, const BatchDev &b, int *bad, const int *pix, int *removed, int first,
                          int *rlist, int *nchanged, int *flag, hipStream_t st)
{
    // free after phase 3: the band ends, stacks and envelopes (every texture has 64 T band ends and T * T
    // entries of the others)
    int *setbad = p.cnt, *chset = p.E;
    unsigned *changed = (unsigned *)p.S;
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
              (const int *)bad, (const int *)setbad, b, changed, chset, nchanged);
    GA_LAUNCH(k_recheck, dim3(1024), dim3(256), 0, st, (const int *)p.vor, pix, b, (const unsigned *)changed,
              (const int *)chset, (const int *)nchanged, bad, flag);
}
