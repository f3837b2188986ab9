/*
 * dcf_basin.hip -- the component tree from the basin graph of the image, without a loop over grey levels.
 *
 * Pixels are ordered by (key, raster index).  Every pixel points to a higher neighbour (its ascent); the
 * pixels that reach the same local maximum (peak) form a basin.  Only a pixel whose higher neighbours are
 * not connected among themselves through higher pixels of its 3x3(x3) surroundings (a saddle) can join two
 * basins, so the graph {peaks, saddles} carries all the tree's branching: its maximum spanning forest is
 * the tree with the pixels between two saddles left out.
 *
 *   k_bs_ascent    one block per tile, keys and halo in LDS: ascents followed to a peak or out of the tile,
 *                  peaks numbered, saddles listed as edges (saddle pixel, neighbour in another part)
 *   k_bs_border    the tile-border pixels' pointers across tiles, shortened
 *   k_bs_edges     edges between the basins of their ends
 *   k_bs_hook / k_bs_merge / k_bs_contract, k_bs_finish
 *                  rounds of Boruvka: every component takes its highest edge; of two that take each other
 *                  the one with the higher peak stays, every other one dies there: branch X ends at the
 *                  grey dval(X) of that edge and continues in the component up(X) that is left after the
 *                  round.  A path along up passes one round per step, so it is O(log peaks) long
 *   k_bs_slots, k_bs_count .. k_bs_sort
 *                  the tree's nodes are the pairs (branch X, key v) that hold pixels: for a branch that is dense
 *                  in its range of keys, one slot per key; for a sparse one, one slot per pixel (a pixel's slot
 *                  is the number of the branch's pixels with higher keys)
 *   k_bs_assign    a pixel of key v lies in the first branch X on the up path of its basin with dval(X) < v:
 *                  its slot.  Then every slot's smallest pixel and pixel count, through bins (k_bs_desc,
 *                  k_bs_bin, k_bs_rest) or, for small images, atomics
 *   k_bs_nodes     nodes numbered along the branches, highest key first: a node's parent is the next one of its
 *                  branch, a branch's last node hangs below the node of grey dval in the branch that holds
 *                  it there (k_bs_link).  The canonical levelroot is the slot's smallest pixel
 *   attributes     each node's own pixels (k_bs_own); a branch's total is the sum of its nodes' and of the
 *                  branches that end on it (k_bs_totals, from the leaves up); each total is added to the node
 *                  its branch hangs below (k_bs_join); the record of a node is a prefix of its branch
 *   k_bs_area, k_bs_parent, k_bs_result, k_bs_records
 *                  everything in raster order
 * The result (canonical parent array, node numbers in raster order of the levelroots, exact integer records)
 * is that of the reference's flooding (tree_flood, src/sources/flood.c:222-247).
 *
 * Measured on the 8192^2 u16 value-noise image: 440 thousand peaks, 2.9 edges per peak, a pixel climbs 3.4
 * branches, 7.5 ms with the filter where a loop over grey levels took 46 (256x320 u8: 0.34 against 4.4); blurred
 * noise with disks has one peak in 12.6 pixels, 1.8 edges per peak: 14.4 ms at 8192^2 u16.
 */
#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <type_traits>
#include <vector>

#include "dcf_internal.h"

#define BS_PEAK 0x80000000u /* a label that is a peak's number; without it, the next pixel of the ascent */
#define BS_NONE 0xFFFFFFFFu
#define BS_EXIT 0x8000u     /* tile-local pointers: the ascent leaves the tile (low bits: direction) */
#define BS_TOP 0x4000u      /* tile-local pointers: a peak */
#define BS_TILE 4096
/* a sparse branch of at most BS_SCAN pixels is searched by looking at every key; a larger one, of at most
 * BS_SORT pixels (what one block sorts in LDS), in its sorted keys.  Builds of 4096^2 u16 disks, u16 noise, f32 noise: 3.50, 3.99, 6.51 ms;
 * with BS_SCAN 16 3.35, 3.88, 6.42, with 128 3.83, 4.25, 6.78; with BS_SORT 2048 3.61, 4.10, 6.64, with 16384 3.54, 4.05, 6.51 */
#define BS_SCAN 48u
#define BS_SORT 8192u

/* ------------------------------------------------------------------------------------------------ */
/* pixel access                                                                                     */
/* ------------------------------------------------------------------------------------------------ */
__device__ __forceinline__ uint32_t bs_key(const ImgView &iv, int64_t p)
{
    if (iv.dtype == DCF_KEY32) return ((const uint32_t *)iv.img)[p];
    const uint32_t v = iv.dtype == DCF_U8 ? ((const uint8_t *)iv.img)[p] : ((const uint16_t *)iv.img)[p];
    /* (the maximum is that of the build: no greater value, unless the caller's image has changed since) */
    const uint32_t gm = iv.invert ? (uint32_t)(*iv.gmax) : 0u;
    return iv.invert ? gm - min(v, gm) : v;
}

/* grey value of pixel p as the reference's float `value` */
__device__ __forceinline__ float bs_grey(const ImgView &iv, int64_t p)
{
    float v;
    if (iv.dtype == DCF_U8) v = (float)((const uint8_t *)iv.img)[p];
    else if (iv.dtype == DCF_U16) v = (float)((const uint16_t *)iv.img)[p];
    else v = ((const float *)iv.img)[p];
    return iv.invert ? *iv.gmax - v : v;
}

/* the images' geometry: one image, or a batch laid out back to back (every image with its own tiles) */
struct BsGeo {
    int W, H, D;
    int64_t n;
    int ntx, nty;
    const BatchImg *bimg;
    int nbatch;
};

struct BsTile {
    int x0, y0, z0, W, H, D;
    int64_t off;
};

template <int TX, int TY, int TZ> __device__ __forceinline__ BsTile bs_tile(const BsGeo &g, int b)
{
    BsTile t;
    int ntx = g.ntx, nty = g.nty;
    t.W = g.W; t.H = g.H; t.D = g.D;
    t.off = 0;
    if (g.bimg) {
        int lo = 0, hi = g.nbatch - 1;
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if ((int)g.bimg[mid].btile0 <= b) lo = mid;
            else hi = mid - 1;
        }
        const BatchImg im = g.bimg[lo];
        t.W = (int)im.W; t.H = (int)im.H; t.D = (int)im.D;
        t.off = (int64_t)im.off;
        b -= (int)im.btile0;
        ntx = (t.W + TX - 1) / TX;
        nty = (t.H + TY - 1) / TY;
    }
    t.x0 = (b % ntx) * TX;
    t.y0 = ((b / ntx) % nty) * TY;
    t.z0 = (b / (ntx * nty)) * TZ;
    return t;
}

/* directions.  2D: the ring E SE S SW W NW N NE, even = edge neighbours; the first four have a larger raster
 * index.  3D: (dz + 1) * 9 + (dy + 1) * 3 + dx + 1, those above 13 have a larger index. */
__device__ __forceinline__ void bs_dir2(int d, int &dx, int &dy)
{
    /* dx + 1 and dy + 1, two bits per direction */
    dx = (int)((0x901Au >> (2 * d)) & 3u) - 1;
    dy = (int)((0x01A9u >> (2 * d)) & 3u) - 1;
}

template <int MODE>
__device__ __forceinline__ typename std::conditional<(MODE < 2), int64_t, int>::type bs_step(int d, int W, int H)
{
    if constexpr (MODE < 2) {
        int dx, dy;
        bs_dir2(d, dx, dy);
        return dx + (int64_t)dy * W;
    } else {
        const int dz = d / 9 - 1, dy = (d / 3) % 3 - 1, dx = d % 3 - 1;
        return dx + dy * W + dz * (W * H);
    }
}

__device__ __forceinline__ uint32_t rot8(uint32_t m, int k) { return ((m << k) | (m >> (8 - k))) & 255u; }

/* 2D: m = the higher pixels of the ring, d = the ascent.  One direction for every connected part of the
 * higher neighbours that does not hold d.  Parts are runs of the ring; with 8-connectivity a missing corner
 * between two present edge neighbours does not cut (they touch each other), with 4-connectivity corners
 * connect but are no neighbours */
template <int MODE> __device__ __forceinline__ uint32_t bs_parts2(uint32_t m, int d)
{
    if constexpr (MODE == 1) {
        const uint32_t e = m & 0x55u;
        const uint32_t f = m | (rot8(e, 1) & rot8(e, 7));
        uint32_t st = f & ~rot8(f, 1);
        if (!(st & (st - 1))) return 0; /* one run (or the whole ring) */
        while ((f >> ((d + 7) & 7)) & 1u) d = (d + 7) & 7;
        return st & ~(1u << d);
    } else {
        const uint32_t e = m & 0x55u, c = m & 0xAAu;
        const uint32_t j = rot8(c, 1) & rot8(e, 2); /* joined to the edge neighbour before, through the corner */
        const uint32_t st = e & ~j;
        if (!(st & (st - 1))) return 0;
        while ((j >> d) & 1u) d = (d + 6) & 7;
        return st & ~(1u << d);
    }
}

/* 3D: the part of the higher neighbours m that holds s, as a fill of the 27 bits.  With 26-connectivity every pair at most
 * one step apart touches.  With 6-connectivity m holds faces and edges (no corners): two faces are joined by the higher
 * edge neighbour between them, which is a step from each. */
template <int MODE> __device__ __forceinline__ uint32_t bs_part3(uint32_t m, int s)
{
    constexpr uint32_t X0 = 0x1249249u, X2 = X0 << 2, Y0 = 7u | (7u << 9) | (7u << 18), Y2 = Y0 << 6;
    uint32_t part = 1u << s, last;
    do {
        last = part;
#pragma unroll
        for (int k = 0; k < 2; k++) {
            if constexpr (MODE == 2) {
                const uint32_t x = ((part & ~X2) << 1) | ((part & ~X0) >> 1), y = ((part & ~Y2) << 3) | ((part & ~Y0) >> 3);
                part |= (x | y | (part << 9) | (part >> 9)) & m;
            } else {
                uint32_t c = part | ((part & ~X2) << 1) | ((part & ~X0) >> 1);
                c |= ((c & ~Y2) << 3) | ((c & ~Y0) >> 3);
                part |= (c | (c << 9) | (c >> 9)) & m;
            }
        }
    } while (part != last);
    return part;
}

template <int MODE> __device__ __forceinline__ uint32_t bs_parts3(uint32_t m, int d)
{
    constexpr uint32_t FACES = (1u << 4) | (1u << 10) | (1u << 12) | (1u << 14) | (1u << 16) | (1u << 22);
    const uint32_t nb = MODE == 2 ? (m & FACES) : m;
    if (!(nb & (nb - 1))) return 0;
    uint32_t rest = nb & ~bs_part3<MODE>(m, d), reps = 0;
    while (rest) {
        const int b = __ffs(rest) - 1;
        reps |= 1u << b;
        rest &= ~bs_part3<MODE>(m, b);
    }
    return reps;
}

/* ------------------------------------------------------------------------------------------------ */
/* basins and saddles                                                                               */
/* ------------------------------------------------------------------------------------------------ */
/* MODE: 0 2D 4-connectivity, 1 2D 8, 2 3D 6, 3 3D 26.  Tiles of 64x64 or 16x16x16, 16 pixels a thread.
 * lab[p] = BS_PEAK | number of p's peak, or the first pixel outside the tile on p's ascent; pval = the
 * peaks' keys; edges = (saddle, neighbour) of every further part; count[0] peaks, count[1] edges (edges
 * beyond ecap are counted, not written). */
template <int MODE>
__global__ __launch_bounds__(256) void k_bs_ascent(ImgView iv, BsGeo g, uint32_t *__restrict__ lab, uint32_t *__restrict__ pval,
                                                   uint2 *__restrict__ edges, uint64_t ecap, unsigned long long *__restrict__ count)
{
    constexpr bool D3 = MODE >= 2;
    constexpr int TX = D3 ? 16 : 64, TY = D3 ? 16 : 64, TZ = D3 ? 16 : 1;
    constexpr int HX = TX + 2, HY = TY + 2, HZ = D3 ? TZ + 2 : 1;
    __shared__ uint32_t kv[HX * HY * HZ]; /* key + 1, 0 outside the image; later the peaks' numbers by tile pixel */
    __shared__ uint16_t to[BS_TILE];
    __shared__ uint32_t npk, nex;
    __shared__ unsigned long long gpk, gex;
    const int tid = threadIdx.x;
    const BsTile t = bs_tile<TX, TY, TZ>(g, blockIdx.x);
    /* pixel numbers are below 2^30; the 2D kernel is a tenth faster with 64-bit ones */
    typedef typename std::conditional<D3, uint32_t, int64_t>::type Pix;
    const Pix off = (Pix)t.off, W = (Pix)t.W, WH = W * (Pix)t.H;
    if (tid == 0) {
        npk = 0;
        nex = 0;
    }
    if constexpr (!D3) {
        for (int i = tid; i < HX * HY; i += 256) {
            const int x = t.x0 + i % HX - 1, y = t.y0 + i / HX - 1;
            const bool in = x >= 0 && x < t.W && y >= 0 && y < t.H;
            kv[i] = in ? bs_key(iv, t.off + x + (int64_t)y * t.W) + 1u : 0u;
        }
    } else {
        /* the thread's next place in the tile with its halo is 256 further: DX columns, DY rows, no slice */
        constexpr int DX = 256 % HX, DY = 256 / HX;
        static_assert(!D3 || DY + 1 < HY, "");
        int x = tid % HX, y = tid / HX, z = 0;
        for (int i = tid; i < HX * HY * HZ; i += 256) {
            const int gx = t.x0 + x - 1, gy = t.y0 + y - 1, gz = t.z0 + z - 1;
            const bool in = (uint32_t)gx < (uint32_t)t.W && (uint32_t)gy < (uint32_t)t.H && (uint32_t)gz < (uint32_t)t.D;
            kv[i] = in ? bs_key(iv, off + (Pix)gx + (Pix)gy * W + (Pix)gz * WH) + 1u : 0u;
            x += DX;
            y += DY;
            if (x >= HX) {
                x -= HX;
                y++;
            }
            if (y >= HY) {
                y -= HY;
                z++;
            }
        }
    }
    __syncthreads();
    uint32_t reps[16];
    uint32_t ex = 0;
#pragma unroll
    for (int i = 0; i < 16; i++) {
        const int l = tid + 256 * i;
        const int lx = l % TX, ly = (l / TX) % TY, lz = l / (TX * TY);
        const int c = D3 ? ((lz + 1) * HY + ly + 1) * HX + lx + 1 : (ly + 1) * HX + lx + 1;
        const uint32_t k0 = kv[c];
        reps[i] = 0;
        if (!k0) continue;
        /* the higher neighbours (equal ones count among those of a larger index), and the highest of them: the ascent, the
         * first direction of equal ones */
        uint32_t m = 0;
        int bd = -1;
        if constexpr (!D3) {
            constexpr int OFF[8] = { 1, HX + 1, HX, HX - 1, -1, -HX - 1, -HX, -HX + 1 };
            uint32_t bk = 0;
#pragma unroll
            for (int d = 0; d < 8; d++) {
                const uint32_t kq = kv[c + OFF[d]];
                const bool hi = d < 4 ? kq >= k0 : kq > k0;
                m |= hi ? 1u << d : 0u;
                if (hi && (MODE == 1 || !(d & 1)) && kq > bk) {
                    bk = kq;
                    bd = d;
                }
            }
            if (bd >= 0) reps[i] = bs_parts2<MODE>(m, bd);
        } else {
            /* from the last direction to the first; top = the key to be reached.  18 or 26 of these are most of the
             * kernel: with this, the fill of bs_part3 and 32-bit pixel numbers 512^3 takes 1.7 ms instead of 3.0 */
            uint32_t top = k0;
#pragma unroll
            for (int d = 26; d >= 0; d--) {
                const int dz = d / 9 - 1, dy = (d / 3) % 3 - 1, dx = d % 3 - 1;
                const int l1 = (dx ? 1 : 0) + (dy ? 1 : 0) + (dz ? 1 : 0);
                if (d == 13) top = max(top, k0 + 1u);
                if (d == 13 || (MODE == 2 && l1 == 3)) {
                    m += m;
                    continue;
                }
                const uint32_t kq = kv[c + (dz * HY + dy) * HX + dx];
                m = m + m + (uint32_t)(d > 13 ? kq >= k0 : kq > k0);
                if ((MODE == 3 || l1 == 1) && kq >= top) {
                    top = kq;
                    bd = d;
                }
            }
            if (bd >= 0) reps[i] = bs_parts3<MODE>(m, bd);
        }
        ex += (uint32_t)__popc(reps[i]);
        uint16_t v = BS_TOP;
        if (bd >= 0) {
            int dx, dy, dz = 0;
            if constexpr (!D3) bs_dir2(bd, dx, dy);
            else {
                dz = bd / 9 - 1;
                dy = (bd / 3) % 3 - 1;
                dx = bd % 3 - 1;
            }
            const int nx = lx + dx, ny = ly + dy, nz = lz + dz;
            const bool in = nx >= 0 && nx < TX && ny >= 0 && ny < TY && nz >= 0 && nz < TZ;
            v = in ? (uint16_t)((nz * TY + ny) * TX + nx) : (uint16_t)(BS_EXIT | (uint32_t)bd);
        }
        to[l] = v;
    }
    const uint32_t eoff = ex ? atomicAdd(&nex, ex) : 0u;
    __syncthreads();
    /* the keys are read: their place takes the peaks' numbers */
    volatile uint16_t *vto = to;
#pragma unroll
    for (int i = 0; i < 16; i++) {
        const int l = tid + 256 * i;
        const int x = t.x0 + l % TX, y = t.y0 + (l / TX) % TY, z = D3 ? t.z0 + l / (TX * TY) : 0;
        if (x >= t.W || y >= t.H || z >= t.D) continue;
        uint32_t v = vto[l];
        if (v == BS_TOP) kv[l] = atomicAdd(&npk, 1u);
        if (v & (BS_EXIT | BS_TOP)) continue;
        /* to the end of the ascent inside the tile (other threads only shorten the pointers they own) */
        for (;;) {
            const uint32_t w = vto[v];
            if (w & (BS_EXIT | BS_TOP)) break;
            v = w;
        }
        vto[l] = (uint16_t)v;
    }
    __syncthreads();
    if (tid == 0) {
        gpk = npk ? atomicAdd(&count[0], (unsigned long long)npk) : 0ull;
        gex = nex ? atomicAdd(&count[1], (unsigned long long)nex) : 0ull;
    }
    __syncthreads();
    uint64_t e = gex + eoff;
#pragma unroll
    for (int i = 0; i < 16; i++) {
        const int l = tid + 256 * i;
        const int x = t.x0 + l % TX, y = t.y0 + (l / TX) % TY, z = D3 ? t.z0 + l / (TX * TY) : 0;
        if (x >= t.W || y >= t.H || z >= t.D) continue;
        const Pix p = off + (Pix)x + (Pix)y * W + (Pix)z * WH;
        uint32_t r = (uint32_t)l, f = to[l];
        if (!(f & (BS_EXIT | BS_TOP))) {
            r = f;
            f = to[r];
        }
        if (f & BS_TOP) {
            const uint32_t id = (uint32_t)gpk + kv[r];
            lab[p] = BS_PEAK | id;
            if (r == (uint32_t)l) pval[id] = bs_key(iv, p);
        } else {
            const int rx = t.x0 + (int)r % TX, ry = t.y0 + ((int)r / TX) % TY, rz = D3 ? t.z0 + (int)r / (TX * TY) : 0;
            lab[p] = (uint32_t)(off + (Pix)rx + (Pix)ry * W + (Pix)rz * WH + (Pix)bs_step<MODE>((int)(f & 31u), t.W, t.H));
        }
        uint32_t m = reps[i];
        while (m) {
            const int d = __ffs(m) - 1;
            m &= m - 1;
            if (e < ecap) edges[e] = make_uint2((uint32_t)p, (uint32_t)(p + (Pix)bs_step<MODE>(d, t.W, t.H)));
            e++;
        }
    }
}

__device__ __forceinline__ uint32_t bs_ld(const uint32_t *a, uint32_t i)
{
    return __hip_atomic_load(&a[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

template <class T> __device__ __forceinline__ T bs_lda(const T *p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
template <class T> __device__ __forceinline__ void bs_sta(T *p, T v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }

/* ---- prefixes in the kernel that needs them (decoupled look-back) ----
 * Blocks take the tiles of an array in order (a ticket: every earlier tile is held by a block that runs or has ended), put
 * their tile's sum into its state word, and sum the words before it back to the nearest one that already holds a whole
 * prefix.  One launch instead of a scan of its own between two kernels; small images are bound by launches.  The words and
 * the ticket start at zero.  state: kind << 62 | value; kind 1 the tile's sum, 2 the sum of all tiles up to it. */
struct BsChain {
    unsigned long long *state;
    uint32_t *ticket;
};

/* the block's tile */
__device__ __forceinline__ uint32_t bs_tile_ticket(const BsChain &ch)
{
    __shared__ uint32_t t;
    if (threadIdx.x == 0) t = atomicAdd(ch.ticket, 1u);
    __syncthreads();
    return t;
}

/* the sum before tile t, to be called by the first wave of a block, once.  sum: the tile's; whole: it already stands for
 * all tiles up to it (a segmented sum that starts inside the tile) */
__device__ __forceinline__ unsigned long long bs_look_back(const BsChain &ch, uint32_t t, unsigned long long sum, bool whole = false)
{
    typedef unsigned long long u64;
    const int lane = threadIdx.x & 63;
    if (lane == 0) bs_sta(&ch.state[t], (u64)(((t == 0 || whole) ? 2ull : 1ull) << 62 | sum));
    u64 before = 0;
    for (int64_t pos = (int64_t)t - 1; pos >= 0; pos -= 64) {
        const int64_t i = pos - lane;
        u64 v = i >= 0 ? bs_lda(&ch.state[i]) : 2ull << 62;
        while (__ballot((v >> 62) == 0))
            if ((v >> 62) == 0) v = bs_lda(&ch.state[i]);
        const u64 m = __ballot((v >> 62) == 2);
        const int stop = m ? __ffsll(m) - 1 : 63;
        u64 x = lane <= stop ? v & ((1ull << 62) - 1) : 0ull;
        for (int o = 32; o > 0; o >>= 1) {
            const uint32_t lo = __shfl_xor((uint32_t)x, o, 64), hi = __shfl_xor((uint32_t)(x >> 32), o, 64);
            x += ((u64)hi << 32) | lo;
        }
        before += x;
        if (m) break;
    }
    if (t != 0 && !whole && lane == 0) bs_sta(&ch.state[t], (u64)(2ull << 62 | (before + sum)));
    return before;
}

/* exclusive prefix of v over the lanes of a wave; sum = the wave's */
__device__ __forceinline__ unsigned long long bs_wave_prefix(unsigned long long v, unsigned long long &sum)
{
    typedef unsigned long long u64;
    const int lane = threadIdx.x & 63;
    u64 x = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t lo = __shfl_up((uint32_t)x, o, 64), hi = __shfl_up((uint32_t)(x >> 32), o, 64);
        if (lane >= o) x += ((u64)hi << 32) | lo;
    }
    sum = ((u64)__shfl((uint32_t)(x >> 32), 63, 64) << 32) | __shfl((uint32_t)x, 63, 64);
    return x - v;
}

/* the peak of pixel p; FRESH: other blocks are shortening the pointers (bs_far), their stores are seen */
template <bool FRESH> __device__ __forceinline__ uint32_t bs_peak(const uint32_t *lab, uint32_t p)
{
    uint32_t v = FRESH ? bs_lda(&lab[p]) : bs_ld(lab, p);
    while (!(v & BS_PEAK)) v = FRESH ? bs_lda(&lab[v]) : bs_ld(lab, v);
    return v & ~BS_PEAK;
}

/* f(pixel) for the border pixels of tile t that this thread of 256 looks after (in 2D the four sides, the corners twice) */
template <bool D3, class F> __device__ __forceinline__ void bs_border_pixels(const BsTile &t, F f)
{
    auto pixel = [&](int lx, int ly, int lz) {
        const int x = t.x0 + lx, y = t.y0 + ly, z = t.z0 + lz;
        if (x < t.W && y < t.H && z < t.D) f((uint32_t)t.off + (uint32_t)(x + y * t.W + z * (t.W * t.H)));
    };
    if constexpr (!D3) {
        const int s = threadIdx.x >> 6, l = threadIdx.x & 63;
        if (s == 0) pixel(l, 0, 0);
        else if (s == 1) pixel(l, 63, 0);
        else if (s == 2) pixel(0, l, 0);
        else pixel(63, l, 0);
    } else {
        for (int i = threadIdx.x; i < BS_TILE; i += 256) {
            const int lx = i & 15, ly = (i >> 4) & 15, lz = i >> 8;
            if (lx == 0 || lx == 15 || ly == 0 || ly == 15 || lz == 0 || lz == 15) pixel(lx, ly, lz);
        }
    }
}

/* The border pixels that k_bs_border leaves short of their peak, by jumps until there are none: the length of a jump doubles
 * with every pass while the blocks advance side by side, so an ascent over the 65536 tiles of a row of 4 million equal pixels
 * takes about a dozen passes.  A pointer only moves along its ascent, so any order of the blocks ends with the same. */
template <bool D3> __device__ __forceinline__ void bs_far(const BsGeo &g, uint32_t *lab, int tiles)
{
    constexpr int T = D3 ? 16 : 64;
    bool left = true;
    while (left) {
        left = false;
        for (int ti = blockIdx.x; ti < tiles; ti += gridDim.x)
            bs_border_pixels<D3>(bs_tile<T, T, D3 ? 16 : 1>(g, ti), [&](uint32_t p) {
                const uint32_t v = bs_lda(&lab[p]);
                if (v & BS_PEAK) return;
                const uint32_t w = bs_lda(&lab[v]);
                bs_sta(&lab[p], w);
                left = left || !(w & BS_PEAK);
            });
    }
}

/* ------------------------------------------------------------------------------------------------ */
/* spanning forest of the basin graph                                                               */
/* ------------------------------------------------------------------------------------------------ */
/* an edge's weight is (key + 1) << 32 | saddle pixel, 0 stands for none.  Edges of equal weight share their saddle, so
 * all of them meet in the saddle's own component: every choice among them is free of cycles. */
struct BsEdges {
    uint64_t *w;
    uint2 *ab;
};

struct BsBor {
    const unsigned long long *count; /* [0] peaks, [1] saddle edges */
    BsEdges e[2];
    uint32_t *ecount;  /* per round: edges */
    uint32_t *deep;    /* per round: a path was longer than BS_WALK, some comp entries lie on the way */
    uint32_t *rcount;  /* per round: components with edges (round 0: all) */
    uint32_t *roots[2];
    uint64_t *best[2]; /* per component: the highest edge's weight */
    uint32_t *hook;    /* the component across it */
    uint32_t *comp;    /* the component after the round (itself: it stays) */
    uint4 *rec;        /* per branch: dval (int, -1: the forest's root), up, and later its slots */
    const uint32_t *pval;
};

__device__ __forceinline__ void bs_best(uint64_t *best, uint32_t c, uint64_t w)
{
    if (__hip_atomic_load(&best[c], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < w)
        atomicMax((unsigned long long *)&best[c], (unsigned long long)w);
}

/* appends to a list for every thread with keep set: one atomic per block; all threads must call it */
__device__ __forceinline__ uint32_t bs_append(bool keep, uint32_t *counter)
{
    __shared__ uint32_t wbase[4], bbase;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const uint64_t m = __ballot(keep);
    __syncthreads();
    if (lane == 0) wbase[w] = (uint32_t)__popcll(m);
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t s = 0;
        for (int i = 0; i < 4; i++) {
            const uint32_t c = wbase[i];
            wbase[i] = s;
            s += c;
        }
        bbase = s ? atomicAdd(counter, s) : 0u;
    }
    __syncthreads();
    return bbase + wbase[w] + (uint32_t)__popcll(m & ((1ull << lane) - 1));
}

template <bool FRESH>
__device__ __forceinline__ void bs_edge_list(const ImgView &iv, const uint32_t *lab, const uint2 *__restrict__ raw, const BsBor &b,
                                             uint64_t ecap)
{
    /* (the host makes room and starts again when the list was too short) */
    const uint32_t E = (uint32_t)min((uint64_t)b.count[1], ecap);
    const uint32_t stride = gridDim.x * 256u;
    for (uint32_t base = blockIdx.x * 256u; base < E; base += stride) {
        const uint32_t i = base + threadIdx.x;
        uint32_t x = 0, y = 0;
        uint64_t w = 0;
        if (i < E) {
            const uint2 r = raw[i];
            x = bs_peak<FRESH>(lab, r.x);
            y = bs_peak<FRESH>(lab, r.y);
            w = ((uint64_t)(bs_key(iv, r.x) + 1u) << 32) | r.x;
        }
        const bool keep = x != y;
        const uint32_t at = bs_append(keep, b.ecount);
        if (keep) {
            b.e[0].w[at] = w;
            b.e[0].ab[at] = make_uint2(x, y);
            bs_best(b.best[0], x, w);
            bs_best(b.best[0], y, w);
        }
    }
}

__global__ __launch_bounds__(256) void k_bs_edges(ImgView iv, const uint32_t *__restrict__ lab, const uint2 *__restrict__ raw,
                                                  BsBor b, uint64_t ecap)
{
    bs_edge_list<false>(iv, lab, raw, b, ecap);
}

/* for images whose border pixels may not be at their peaks (others have had k_bs_init) */
template <bool D3>
__global__ __launch_bounds__(256) void k_bs_edges_far(ImgView iv, BsGeo g, uint32_t *lab, const uint32_t *__restrict__ more, int tiles,
                                                      const uint2 *__restrict__ raw, BsBor b, uint64_t ecap)
{
    if (*more) {
        bs_far<D3>(g, lab, tiles);
        bs_edge_list<true>(iv, lab, raw, b, ecap);
    } else bs_edge_list<false>(iv, lab, raw, b, ecap);
}

__device__ __forceinline__ void bs_init(const BsBor &b, uint32_t i)
{
    b.best[0][i] = 0;
    b.best[1][i] = 0;
    b.comp[i] = i;
    b.rec[i] = make_uint4(0xFFFFFFFFu, i, 0u, 0u);
}

template <bool D3>
__global__ __launch_bounds__(256) void k_bs_init(BsGeo g, uint32_t *lab, const uint32_t *__restrict__ more, int tiles, BsBor b)
{
    if (*more) bs_far<D3>(g, lab, tiles);
    const uint32_t G = (uint32_t)b.count[0];
    for (uint32_t i = blockIdx.x * 256u + threadIdx.x; i < G; i += gridDim.x * 256u) bs_init(b, i);
}

/* Ascents enter a tile at its border pixels: their pointers are shortened by up to 16 steps a launch.  One launch covers the 15
 * tiles that ascents cross in ordinary images of up to 2^22 pixels; three, in larger ones, cover at least 4096 tiles.
 * more[round] is set when a pointer is still not at its peak (a wide plateau, a long thin image): bs_far does the rest, in
 * a kernel that is there anyway.  A launch after one that left none returns at once.
 * init: also the start of the forest's arrays (their launch saved). */
template <int MODE>
__global__ __launch_bounds__(256) void k_bs_border(BsGeo g, uint32_t *lab, uint32_t *more, int round, BsBor b, int init)
{
    constexpr bool D3 = MODE >= 2;
    constexpr int TX = D3 ? 16 : 64, TY = D3 ? 16 : 64, TZ = D3 ? 16 : 1;
    if (init) {
        const uint32_t G = (uint32_t)b.count[0];
        for (uint32_t i = blockIdx.x * 256u + threadIdx.x; i < G; i += gridDim.x * 256u) bs_init(b, i);
    }
    if (round > 0 && more[round - 1] == 0) return;
    const BsTile t = bs_tile<TX, TY, TZ>(g, blockIdx.x);
    bool left = false;
    bs_border_pixels<D3>(t, [&](uint32_t p) {
        uint32_t v = bs_ld(lab, p);
        if (v & BS_PEAK) return;
        for (int s = 0; s < 16 && !(v & BS_PEAK); s++) v = bs_ld(lab, v);
        left = left || !(v & BS_PEAK);
        bs_sta(&lab[p], v);
    });
    /* one thread of a block looks past the caches before it stores (one store per wave, all on one word, were 6.5 of the 6.7 ms of
     * this kernel for a row of 2^22 equal pixels) */
    if (__syncthreads_or(left) && threadIdx.x == 0 && bs_lda(&more[round]) == 0) bs_sta(&more[round], 1u);
}

__global__ __launch_bounds__(256) void k_bs_hook(BsBor b, int round)
{
    const int q = round & 1;
    const uint32_t E = b.ecount[round];
    for (uint32_t i = blockIdx.x * 256u + threadIdx.x; i < E; i += gridDim.x * 256u) {
        const uint64_t w = b.e[q].w[i];
        const uint2 ab = b.e[q].ab[i];
        if (b.best[q][ab.x] == w) b.hook[ab.x] = ab.y;
        if (b.best[q][ab.y] == w) b.hook[ab.y] = ab.x;
    }
}

/* component x stays a root in this round: it has no edge, or it and the component it takes take each other
 * over edges of one weight and x has the higher peak */
template <class LD64, class LD32, class PV>
__device__ __forceinline__ bool bs_stays(uint32_t x, uint32_t &t, LD64 ldbest, LD32 ldhook, PV peak)
{
    const uint64_t w = ldbest(x);
    if (!w) return true;
    t = ldhook(x);
    if (ldbest(t) != w || ldhook(t) != x) return false;
    const uint32_t px = peak(x), pt = peak(t);
    return px > pt || (px == pt && x > t);
}

/* Paths of components that take each other.  On noise and smooth images they are one or two steps long, 15 at most on
 * the images of the benchmark; where the saddles' order follows the image (equal greys: a binary image, a halftone; or a
 * texture on a ramp) they are as long as the image (2048^2 checkerboard: 2.1 million components, 1023 steps each).  A thread
 * walks BS_WALK steps; paths that go on are resolved by jumps over the comp entries, which double with every step while
 * the threads advance side by side, and are right in any order (an entry only moves along its path to its end).  Whole
 * builds at 8192^2 u8: checkerboard 12.3 ms, halftone 8.5, uniform noise 13.2. */
#define BS_WALK 24

/* comp[x] to the component that stays, and the end of x's branch; x died in this round */
__device__ __forceinline__ bool bs_jump(uint32_t *comp, uint4 *rec, uint32_t x)
{
    const uint32_t c = bs_lda(&comp[x]), r = bs_lda(&comp[c]);
    if (r == c) return false;
    bs_sta(&comp[x], r);
    rec[x].y = r;
    return true;
}

__device__ __forceinline__ uint32_t bs_end(const uint32_t *comp, uint32_t x)
{
    for (;;) {
        const uint32_t c = bs_lda(&comp[x]);
        if (c == x) return x;
        x = c;
    }
}

__global__ __launch_bounds__(256) void k_bs_merge(BsBor b, int round)
{
    const int q = round & 1;
    const uint32_t R = round == 0 ? (uint32_t)b.count[0] : b.rcount[round];
    const uint64_t *best = b.best[q];
    const uint32_t *hook = b.hook;
    auto l64 = [&](uint32_t i) { return best[i]; };
    auto l32 = [&](uint32_t i) { return hook[i]; };
    auto peak = [&](uint32_t i) { return b.pval[i]; };
    const uint32_t stride = gridDim.x * 256u;
    for (uint32_t base = blockIdx.x * 256u; base < R; base += stride) {
        const uint32_t i = base + threadIdx.x;
        bool live = false;
        uint32_t x = 0;
        if (i < R) {
            x = round == 0 ? i : b.roots[q][i];
            const uint64_t w = best[x];
            uint32_t r = x, t = 0;
            int steps = 0;
            while (!bs_stays(r, t, l64, l32, peak)) {
                r = t;
                if (++steps == BS_WALK) break;
            }
            if (steps == BS_WALK && bs_lda(&b.deep[round]) == 0) bs_sta(&b.deep[round], 1u);
            b.comp[x] = r;
            if (r != x) {
                b.rec[x].x = (uint32_t)(w >> 32) - 1u;
                b.rec[x].y = r;
            } else {
                live = w != 0;
                b.best[1 - q][x] = 0;
            }
        }
        const uint32_t at = bs_append(live, &b.rcount[round + 1]);
        if (live) b.roots[1 - q][at] = x;
    }
}

/* Edges to the components of the next round.  Two large components touch along many saddles and only the highest can
 * matter: a block takes BS_CHUNK edges (neighbours in the list are neighbours in the image) and keeps, through a table in
 * LDS, the highest of each pair of components; an edge that finds no place in the table is kept. */
#define BS_CHUNK 1024
__global__ __launch_bounds__(256) void k_bs_contract(BsBor b, int round)
{
    constexpr int TAB = 1024, PER = BS_CHUNK / 256;
    __shared__ unsigned long long pair[TAB], high[TAB];
    __shared__ uint32_t wsum[4], bbase;
    const int q = round & 1;
    const uint32_t E = b.ecount[round];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const bool deep = b.deep[round] != 0;
    if (deep) {
        const uint32_t R = round == 0 ? (uint32_t)b.count[0] : b.rcount[round];
        bool more = true;
        while (more) {
            more = false;
            for (uint32_t i = blockIdx.x * 256u + threadIdx.x; i < R; i += gridDim.x * 256u)
                more = bs_jump(b.comp, b.rec, round == 0 ? i : b.roots[q][i]) || more;
        }
    }
    for (uint32_t base = blockIdx.x * BS_CHUNK; base < E; base += gridDim.x * BS_CHUNK) {
        for (int i = threadIdx.x; i < TAB; i += 256) {
            pair[i] = ~0ull;
            high[i] = 0ull;
        }
        __syncthreads();
        uint2 ab[PER];
        uint64_t w[PER];
        int at[PER];
#pragma unroll
        for (int k = 0; k < PER; k++) {
            const uint32_t i = base + threadIdx.x + 256u * k;
            w[k] = 0;
            ab[k] = make_uint2(0, 0);
            if (i < E) {
                ab[k] = b.e[q].ab[i];
                w[k] = b.e[q].w[i];
            }
        }
        if (deep) {
            /* another block may still be at its entries */
            for (int k = 0; k < PER; k++)
                if (w[k]) ab[k] = make_uint2(bs_end(b.comp, ab[k].x), bs_end(b.comp, ab[k].y));
        } else {
#pragma unroll
            for (int k = 0; k < PER; k++)
                if (w[k]) {
                    ab[k].x = b.comp[ab[k].x];
                    ab[k].y = b.comp[ab[k].y];
                }
        }
#pragma unroll
        for (int k = 0; k < PER; k++) {
            at[k] = -1;
            if (!w[k]) continue;
            if (ab[k].x == ab[k].y) {
                w[k] = 0;
                continue;
            }
            const unsigned long long id = ((unsigned long long)min(ab[k].x, ab[k].y) << 32) | max(ab[k].x, ab[k].y);
            unsigned long long h = id * 0x9E3779B97F4A7C15ull;
            uint32_t j = (uint32_t)(h >> 54); /* 10 bits */
            for (int i = 0; i < 8 && at[k] < 0; i++) {
                const unsigned long long o = atomicCAS(&pair[j], ~0ull, id);
                if (o == ~0ull || o == id) at[k] = (int)j;
                j = (j + 1) & (TAB - 1);
            }
            if (at[k] >= 0) atomicMax(&high[at[k]], (unsigned long long)w[k]);
        }
        __syncthreads();
        uint32_t mine = 0;
#pragma unroll
        for (int k = 0; k < PER; k++) {
            if (w[k] && at[k] >= 0 && high[at[k]] != w[k]) w[k] = 0;
            mine += w[k] != 0;
        }
        /* the block's places in the next list: prefix of the threads' counts, one atomic */
        uint32_t pre = mine;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t u = __shfl_up(pre, o, 64);
            if (lane >= o) pre += u;
        }
        if (lane == 63) wsum[wv] = pre;
        __syncthreads();
        if (threadIdx.x == 0) {
            uint32_t t = 0;
            for (int i = 0; i < 4; i++) {
                const uint32_t c = wsum[i];
                wsum[i] = t;
                t += c;
            }
            bbase = t ? atomicAdd(&b.ecount[round + 1], t) : 0u;
        }
        __syncthreads();
        uint32_t o = bbase + wsum[wv] + pre - mine;
#pragma unroll
        for (int k = 0; k < PER; k++)
            if (w[k]) {
                b.e[1 - q].w[o] = w[k];
                b.e[1 - q].ab[o] = ab[k];
                o++;
                bs_best(b.best[1 - q], ab[k].x, w[k]);
                bs_best(b.best[1 - q], ab[k].y, w[k]);
            }
        __syncthreads();
    }
}

/* The remaining rounds in one block: a launch costs more than a round of a few thousand edges.  With at most
 * BS_FC components and BS_FE edges per thread the components' arrays are in LDS and a thread reads only its own edges
 * from memory.  More are first brought down in memory; there, what one phase writes another thread reads in the next past this CU's L1, so
 * those accesses are agent-scope. */
#define BS_FT 1024
#define BS_FC 8192
#define BS_FE 32
#define BS_FLDS (BS_FC * (8 + 4 + 2 + 2)) /* bytes: 128 KB of the CU's 160 */
__global__ __launch_bounds__(BS_FT) void k_bs_finish(BsBor b, int round)
{
    extern __shared__ unsigned long long lds[];
    unsigned long long *best = lds;
    uint32_t *pv = (uint32_t *)(best + BS_FC);
    uint16_t *hook = (uint16_t *)(pv + BS_FC), *comp = hook + BS_FC;
    __shared__ uint32_t s_e, s_r;
    uint32_t E = b.ecount[round], R = round == 0 ? (uint32_t)b.count[0] : b.rcount[round];
    bool first = round == 0;
    int q = round & 1;
    const uint32_t tid = threadIdx.x;
    while (E && (E > BS_FT * BS_FE || R > BS_FC)) {
        for (uint32_t i = tid; i < E; i += BS_FT) {
            const uint64_t w = bs_lda(&b.e[q].w[i]);
            const uint64_t ab = bs_lda((const uint64_t *)&b.e[q].ab[i]);
            const uint32_t x = (uint32_t)ab, y = (uint32_t)(ab >> 32);
            if (bs_lda(&b.best[q][x]) == w) bs_sta(&b.hook[x], y);
            if (bs_lda(&b.best[q][y]) == w) bs_sta(&b.hook[y], x);
        }
        if (tid == 0) s_e = s_r = 0;
        __threadfence();
        __syncthreads();
        auto l64 = [&](uint32_t i) { return bs_lda(&b.best[q][i]); };
        auto l32 = [&](uint32_t i) { return bs_lda(&b.hook[i]); };
        auto peak = [&](uint32_t i) { return b.pval[i]; };
        bool more = false;
        for (uint32_t i = tid; i < R; i += BS_FT) {
            const uint32_t x = first ? i : bs_lda(&b.roots[q][i]);
            const uint64_t w = l64(x);
            uint32_t r = x, t = 0;
            int steps = 0;
            while (!bs_stays(r, t, l64, l32, peak)) {
                r = t;
                if (++steps == BS_WALK) break;
            }
            more = more || steps == BS_WALK;
            bs_sta(&b.comp[x], r);
            if (r != x) {
                b.rec[x].x = (uint32_t)(w >> 32) - 1u;
                b.rec[x].y = r;
            } else {
                bs_sta(&b.best[1 - q][x], (uint64_t)0);
                if (w) bs_sta(&b.roots[1 - q][atomicAdd(&s_r, 1u)], x);
            }
        }
        __threadfence();
        while (__syncthreads_or(more)) {
            more = false;
            for (uint32_t i = tid; i < R; i += BS_FT)
                more = bs_jump(b.comp, b.rec, first ? i : bs_lda(&b.roots[q][i])) || more;
            __threadfence();
        }
        for (uint32_t i = tid; i < E; i += BS_FT) {
            const uint64_t ab = bs_lda((const uint64_t *)&b.e[q].ab[i]);
            const uint32_t x = bs_lda(&b.comp[(uint32_t)ab]), y = bs_lda(&b.comp[(uint32_t)(ab >> 32)]);
            if (x == y) continue;
            const uint64_t w = bs_lda(&b.e[q].w[i]);
            const uint32_t at = atomicAdd(&s_e, 1u);
            bs_sta(&b.e[1 - q].w[at], w);
            bs_sta((uint64_t *)&b.e[1 - q].ab[at], ((uint64_t)y << 32) | x);
            bs_best(b.best[1 - q], x, w);
            bs_best(b.best[1 - q], y, w);
        }
        __threadfence();
        __syncthreads();
        E = s_e;
        R = s_r;
        first = false;
        q = 1 - q;
        __syncthreads();
    }
    if (!E) return;
    /* components numbered by their place in the list */
    for (uint32_t i = tid; i < R; i += BS_FT) {
        const uint32_t x = first ? i : bs_lda(&b.roots[q][i]);
        pv[i] = b.pval[x];
        best[i] = 0;
        comp[i] = (uint16_t)i;
        if (!first) bs_sta(&b.comp[x], i);
    }
    __threadfence();
    __syncthreads();
    /* every thread keeps to its own edges: their weights, and their ends as two 16-bit places (or DEAD) in the list
     * that is free */
    constexpr uint32_t DEAD = 0xFFFFFFFFu;
    const uint64_t *ew = b.e[q].w;
    uint32_t *ends = (uint32_t *)b.e[1 - q].ab;
    for (uint32_t i = tid; i < E; i += BS_FT) {
        const uint64_t ab = bs_lda((const uint64_t *)&b.e[q].ab[i]);
        uint32_t x = (uint32_t)ab, y = (uint32_t)(ab >> 32);
        if (!first) {
            x = bs_lda(&b.comp[x]);
            y = bs_lda(&b.comp[y]);
        }
        ends[i] = (y << 16) | x;
    }
    volatile uint16_t *vcomp = comp;
    auto l64 = [&](uint32_t i) { return (uint64_t)best[i]; };
    auto l32 = [&](uint32_t i) { return (uint32_t)hook[i]; };
    auto peak = [&](uint32_t i) { return pv[i]; };
    for (;;) {
        /* every edge to its components; those left inside one are dropped */
        bool any = false;
#pragma unroll 4
        for (uint32_t i = tid; i < E; i += BS_FT) {
            const uint32_t e = ends[i];
            if (e == DEAD) continue;
            const uint32_t x = comp[e & 0xFFFFu], y = comp[e >> 16];
            ends[i] = x == y ? DEAD : (y << 16) | x;
            if (x == y) continue;
            any = true;
            const unsigned long long w = bs_lda(&ew[i]);
            atomicMax(&best[x], w);
            atomicMax(&best[y], w);
        }
        if (!__syncthreads_or(any)) break;
        bool more = false;
#pragma unroll 4
        for (uint32_t i = tid; i < E; i += BS_FT) {
            const uint32_t e = ends[i];
            if (e == DEAD) continue;
            const uint32_t x = e & 0xFFFFu, y = e >> 16;
            const uint64_t w = bs_lda(&ew[i]);
            if (best[x] == w) hook[x] = (uint16_t)y;
            if (best[y] == w) hook[y] = (uint16_t)x;
        }
        __syncthreads();
        for (uint32_t i = tid; i < R; i += BS_FT) {
            const uint64_t w = best[i];
            if (!w) continue; /* dead, or done */
            uint32_t r = i, t = 0;
            int steps = 0;
            while (!bs_stays(r, t, l64, l32, peak)) {
                r = t;
                if (++steps == BS_WALK) break;
            }
            if (r == i) continue;
            more = more || steps == BS_WALK;
            vcomp[i] = (uint16_t)r;
            const uint32_t x = first ? i : bs_lda(&b.roots[q][i]);
            b.rec[x].x = (uint32_t)(w >> 32) - 1u;
            b.rec[x].y = first ? r : bs_lda(&b.roots[q][r]);
        }
        while (__syncthreads_or(more)) {
            more = false;
            for (uint32_t i = tid; i < R; i += BS_FT) {
                if (!best[i]) continue;
                const uint32_t s = vcomp[i], r = vcomp[s];
                if (r == s) continue;
                vcomp[i] = (uint16_t)r;
                const uint32_t x = first ? i : bs_lda(&b.roots[q][i]);
                b.rec[x].y = first ? r : bs_lda(&b.roots[q][r]);
                more = true;
            }
        }
        for (uint32_t i = tid; i < R; i += BS_FT) best[i] = 0;
        __syncthreads();
    }
}

/* ------------------------------------------------------------------------------------------------ */
/* branches, slots                                                                                  */
/* ------------------------------------------------------------------------------------------------ */
/* the branch of key v on the up path of branch x */
__device__ __forceinline__ uint32_t bs_climb(const uint4 *__restrict__ rec, uint32_t x, uint32_t v, uint4 &r)
{
    r = rec[x];
    while ((int32_t)r.x >= (int32_t)v) {
        x = r.y;
        r = rec[x];
    }
    return x;
}

/* Slots.  A dense branch (at least one pixel for two keys of its range, or more than BS_SORT pixels) has one slot per
 * key: record z = first slot + peak key, w = 0.  A sparse one has one per pixel: z = first slot, w = pixels, its keys in
 * skey (sorted from the highest down when there are more than BS_SCAN).  Ranks of a float image can spread a large
 * branch over millions of keys; it is cut into pieces of 2^piece keys, each dense (with more than BS_SORT pixels) or sparse
 * by itself: z = first piece, w = BS_PIECES, and prec holds the pieces' z and w.  piece is BS_PIECE, or more where that makes
 * more than a piece for 64 pixels: many hills over the whole range of keys would have n^2 / 2^27 pieces, more than 32
 * bits count from 2^29 pixels on. */
#define BS_PIECE 14
#define BS_PIECES 0xFFFFFFFFu
struct BsSlots {
    const uint32_t *pval;
    const uint32_t *skey;
    const uint2 *prec;
    int piece;
};

__device__ __forceinline__ uint32_t bs_slot(const uint4 &r, uint32_t x, uint32_t v, const BsSlots &t)
{
    uint32_t z = r.z, w = r.w;
    if (w == 0) return z - v;
    if (w == BS_PIECES) {
        const uint2 q = t.prec[z + ((t.pval[x] - v) >> t.piece)];
        z = q.x;
        w = q.y;
        if (w == 0) return z - v;
    }
    uint32_t higher = 0;
    if (w <= BS_SCAN) {
        for (uint32_t i = 0; i < w; i++) higher += t.skey[z + i] > v;
    } else {
        uint32_t lo = 0, hi = w;
        while (lo < hi) {
            const uint32_t mid = (lo + hi) >> 1;
            if (t.skey[z + mid] > v) lo = mid + 1;
            else hi = mid;
        }
        higher = lo;
    }
    return z + higher;
}

/* keys of branch x's range */
__device__ __forceinline__ uint64_t bs_span(const uint4 &r, uint32_t pv) { return (uint64_t)((int64_t)pv - (int64_t)(int32_t)r.x); }

/* the kind of a branch of s keys and c pixels: 0 dense, 1 sparse, 2 in pieces (a branch too large to be sorted, of more
 * than loose keys per pixel).  loose is 8 while eight slots per pixel fit 31 bits: then the branches of 16-bit keys are
 * never cut, since more than BS_SORT pixels have at least an eighth of 65536 keys. */
__device__ __forceinline__ int bs_kind(uint64_t s, uint32_t c, uint32_t loose)
{
    if (s <= (uint64_t)min(loose, 2u) * c) return 0;
    if (c <= BS_SORT) return 1;
    return s > (uint64_t)loose * c ? 2 : 0;
}

/* *sum grows by the v of a block's 256 threads */
__device__ __forceinline__ void bs_block_add(unsigned long long v, unsigned long long *sum)
{
    __shared__ unsigned long long part[4];
    for (int o = 32; o > 0; o >>= 1) {
        const uint32_t lo = __shfl_xor((uint32_t)v, o, 64), hi = __shfl_xor((uint32_t)(v >> 32), o, 64);
        v += ((unsigned long long)hi << 32) | lo;
    }
    __syncthreads();
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        const unsigned long long b = part[0] + part[1] + part[2] + part[3];
        if (b) atomicAdd(sum, b);
    }
}

/* the slots of every branch when all are dense: first slot (base, one past the last branch too) and record, all their
 * slots (total[0]); and the branches' counters for the attribute pass start at zero */
__global__ __launch_bounds__(256) void k_bs_slots(uint4 *__restrict__ rec, const uint32_t *__restrict__ pval, uint32_t *__restrict__ base,
                                                  const unsigned long long *__restrict__ count, unsigned long long *__restrict__ total,
                                                  BsChain ch, uint32_t *__restrict__ nch, uint32_t *__restrict__ done)
{
    typedef unsigned long long u64;
    __shared__ u64 wsum[4], carry;
    const uint32_t G = (uint32_t)count[0];
    const uint32_t t = bs_tile_ticket(ch);
    if ((uint64_t)t * 1024u > G) return;
    const uint32_t x0 = t * 1024u + threadIdx.x * 4u;
    const int w = threadIdx.x >> 6;
    u64 s[4], v = 0, sum;
    uint4 r[4];
    uint32_t pv[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        r[i] = make_uint4(0, 0, 0, 0);
        pv[i] = 0;
        s[i] = 0;
        if (x0 + i < G) {
            r[i] = rec[x0 + i];
            pv[i] = pval[x0 + i];
            s[i] = bs_span(r[i], pv[i]);
        }
        v += s[i];
    }
    u64 pre = bs_wave_prefix(v, sum);
    if ((threadIdx.x & 63) == 0) wsum[w] = sum;
    __syncthreads();
    const u64 all = wsum[0] + wsum[1] + wsum[2] + wsum[3];
    if (w == 0) {
        const u64 before = bs_look_back(ch, t, all);
        if (threadIdx.x == 0) carry = before;
    }
    __syncthreads();
    pre += carry;
    for (int k = 0; k < w; k++) pre += wsum[k];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const uint32_t x = x0 + i;
        if (x <= G) base[x] = (uint32_t)pre;
        if (x == G) *total = pre;
        if (x < G) {
            rec[x] = make_uint4(r[i].x, r[i].y, (uint32_t)pre + pv[i], 0u);
            nch[x] = 0;
            done[x] = 0;
        }
        pre += s[i];
    }
}

/* slots of every branch by its pixel count, and their sum (sum[0]; without those of the pieces, which are known later); the
 * branches' pieces of 2^piece keys, and their sum (sum[2]) */
__global__ __launch_bounds__(256) void k_bs_range(const uint4 *__restrict__ rec, const uint32_t *__restrict__ pval,
                                                  const uint32_t *__restrict__ bcnt, uint32_t *__restrict__ size,
                                                  uint32_t *__restrict__ pieces, uint32_t loose, int piece, uint32_t G,
                                                  unsigned long long *__restrict__ sum)
{
    uint64_t v = 0, u = 0;
    for (uint64_t x = (uint64_t)blockIdx.x * 256u + threadIdx.x; x <= G; x += (uint64_t)gridDim.x * 256u) {
        uint64_t s = 0, np = 0;
        if (x < G) {
            s = bs_span(rec[x], pval[x]);
            const uint32_t c = bcnt[x];
            const int kind = bs_kind(s, c, loose);
            if (kind == 2) np = (s + (1ull << piece) - 1) >> piece;
            if (kind) s = kind == 1 ? c : 0u;
        }
        v += s;
        u += np;
        size[x] = (uint32_t)s;
        pieces[x] = (uint32_t)np;
    }
    bs_block_add(v, sum);
    bs_block_add(u, sum + 2);
}

/* slots of every piece, and their sum */
__global__ __launch_bounds__(256) void k_bs_piece_size(const uint32_t *__restrict__ pcnt, uint32_t *__restrict__ size, uint32_t NP,
                                                       int piece, unsigned long long *__restrict__ sum)
{
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    const uint32_t c = i < NP ? pcnt[i] : 0u, s = c > BS_SORT ? 1u << piece : c;
    if (i <= NP) size[i] = s;
    bs_block_add(s, sum);
}

/* slots of the branches in pieces (pofs: first piece of every branch, psum: slots before every piece) */
__global__ __launch_bounds__(256) void k_bs_piece_sum(const uint32_t *__restrict__ pofs, const uint32_t *__restrict__ psum,
                                                      uint32_t *__restrict__ size, uint32_t G)
{
    const uint32_t x = blockIdx.x * 256u + threadIdx.x;
    if (x < G && pofs[x + 1] > pofs[x]) size[x] = psum[pofs[x + 1]] - psum[pofs[x]];
}

/* the pieces' records; those to be sorted go to the list mid (first slot, pixels) */
__global__ __launch_bounds__(256) void k_bs_piece_base(const uint32_t *__restrict__ pval, const uint32_t *__restrict__ pofs,
                                                       const uint32_t *__restrict__ psum, const uint32_t *__restrict__ pcnt,
                                                       const uint32_t *__restrict__ base, uint2 *__restrict__ prec,
                                                       uint2 *__restrict__ mid, uint32_t *__restrict__ nmid, int piece, uint32_t NP,
                                                       uint32_t G)
{
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i >= NP) return;
    /* the branch: the last one whose first piece is at or before i (branches without pieces start where the next does) */
    uint32_t lo = 0, hi = G - 1;
    while (lo < hi) {
        const uint32_t m = (lo + hi + 1) >> 1;
        if (pofs[m] <= i) lo = m;
        else hi = m - 1;
    }
    const uint32_t c = pcnt[i], b = base[lo] + psum[i] - psum[pofs[lo]];
    const uint32_t top = pval[lo] - ((i - pofs[lo]) << piece);
    prec[i] = c > BS_SORT ? make_uint2(b + top, 0u) : make_uint2(b, c);
    if (c > BS_SCAN && c <= BS_SORT) mid[atomicAdd(nmid, 1u)] = make_uint2(b, c);
}

/* the records' z and w from base[x], the branch's first slot; sparse branches to be sorted go to mid */
__global__ __launch_bounds__(256) void k_bs_base(uint4 *__restrict__ rec, const uint32_t *__restrict__ pval, const uint32_t *__restrict__ bcnt,
                                                 const uint32_t *__restrict__ base, const uint32_t *__restrict__ pofs, uint32_t loose,
                                                 uint2 *__restrict__ mid, uint32_t *__restrict__ nmid, uint32_t G)
{
    const uint32_t x = blockIdx.x * 256u + threadIdx.x;
    bool sort = false;
    uint32_t c = 0;
    if (x < G) {
        const uint4 r = rec[x];
        const uint32_t pv = pval[x];
        c = bcnt[x];
        const int kind = bs_kind(bs_span(r, pv), c, loose);
        const uint32_t b = base[x];
        rec[x] = make_uint4(r.x, r.y, kind == 0 ? b + pv : (kind == 1 ? b : pofs[x]), kind == 0 ? 0u : (kind == 1 ? c : BS_PIECES));
        sort = kind == 1 && c > BS_SCAN;
    }
    const uint32_t at = bs_append(sort, nmid);
    if (sort) mid[at] = make_uint2(base[x], c);
}

/* the lanes of a wave hold pixels of one tile in raster order: head = the first lane of each run of equal values
 * in one tile row, len = the run's lanes (for its head), at = the lane of its head */
__device__ __forceinline__ void bs_runs(bool valid, uint32_t v, bool row, bool &head, uint32_t &len, int &at)
{
    const int lane = threadIdx.x & 63;
    const uint64_t vm = __ballot(valid);
    const uint32_t pv = __shfl_up(v, 1, 64);
    head = valid && (lane == 0 || row || pv != v || !((vm >> (lane - 1)) & 1ull));
    const uint64_t hm = __ballot(head);
    const uint64_t above = lane == 63 ? 0ull : (hm | ~vm) >> (lane + 1);
    len = above ? (uint32_t)__ffsll((unsigned long long)above) : (uint32_t)(64 - lane);
    at = 63 - __clzll((long long)(hm & (lane == 63 ? ~0ull : ((2ull << lane) - 1))));
}

/* ---- per-tile tables ----
 * A branch, node or slot collects pixels from all over the image, and the big ones would take one atomic on the same word
 * per run of pixels (thousands of atomics on one word cost about 50 ns each; 114 ms on the background's slots of the
 * 512^3 u8 volume).  Each block therefore first collects its tile in a table in LDS (open addressing, a few probes; an
 * item that finds no place is handled by itself). */
#define BS_TAB 2048
#define BS_PROBES 12

__device__ __forceinline__ int bs_find(uint32_t *key, uint32_t v)
{
    uint32_t h = (v * 2654435761u) >> 21; /* 11 bits */
    for (int i = 0; i < BS_PROBES; i++) {
        const uint32_t k = atomicCAS(&key[h], BS_NONE, v);
        if (k == BS_NONE || k == v) return (int)h;
        h = (h + 1) & (BS_TAB - 1);
    }
    return -1;
}

template <bool D3> struct BsShape3 {
    static constexpr int TX = D3 ? 16 : 64, TY = D3 ? 16 : 64, TZ = D3 ? 16 : 1;
};

/* the tile's pixels, and the pixels of the tiles before it (tiles in order: n pixels in all) */
template <bool D3> __device__ __forceinline__ uint32_t bs_tile_pixels(const BsTile &t, uint32_t &before)
{
    constexpr int TX = BsShape3<D3>::TX, TY = BsShape3<D3>::TY, TZ = BsShape3<D3>::TZ;
    const int64_t dx = min(TX, t.W - t.x0), dy = min(TY, t.H - t.y0), dz = min(TZ, t.D - t.z0);
    before = (uint32_t)(t.off + (int64_t)t.z0 * t.W * t.H + (int64_t)t.y0 * t.W * dz + (int64_t)t.x0 * dy * dz);
    return (uint32_t)(dx * dy * dz);
}

/* local pixel l of tile t: its pixel, or -1 outside the image */
template <bool D3> __device__ __forceinline__ int bs_at(const BsTile &t, int l)
{
    constexpr int TX = BsShape3<D3>::TX, TY = BsShape3<D3>::TY;
    const int x = t.x0 + l % TX, y = t.y0 + (l / TX) % TY, z = D3 ? t.z0 + l / (TX * TY) : 0;
    if (x >= t.W || y >= t.H || z >= t.D) return -1;
    return (int)t.off + x + y * t.W + z * (t.W * t.H); /* below 2^30 */
}

/* v, which the compiler takes for another value: what is computed from it again is not kept in registers meanwhile */
__device__ __forceinline__ int bs_opaque(int v)
{
    asm volatile("" : "+v"(v));
    return v;
}

#define BS_AHEAD 4 /* pixels a thread follows side by side: their loads are in flight together */

/* the branches of BS_AHEAD pixels from their labels, the chains of loads side by side */
__device__ __forceinline__ void bs_branches(const uint4 *__restrict__ rec, const uint32_t *lab, const int (&p)[BS_AHEAD],
                                            const uint32_t (&v)[BS_AHEAD], uint32_t (&x)[BS_AHEAD], uint4 (&r)[BS_AHEAD])
{
#pragma unroll
    for (int j = 0; j < BS_AHEAD; j++) x[j] = p[j] >= 0 ? bs_ld(lab, (uint32_t)p[j]) : BS_PEAK;
    bool more = true;
    while (more) {
        more = false;
#pragma unroll
        for (int j = 0; j < BS_AHEAD; j++)
            if (!(x[j] & BS_PEAK)) {
                x[j] = bs_ld(lab, x[j]);
                more = more || !(x[j] & BS_PEAK);
            }
    }
#pragma unroll
    for (int j = 0; j < BS_AHEAD; j++) {
        x[j] &= ~BS_PEAK;
        r[j] = rec[x[j]];
    }
    more = true;
    while (more) {
        more = false;
#pragma unroll
        for (int j = 0; j < BS_AHEAD; j++)
            if (p[j] >= 0 && (int32_t)r[j].x >= (int32_t)v[j]) {
                x[j] = r[j].y;
                r[j] = rec[x[j]];
                more = more || (int32_t)r[j].x >= (int32_t)v[j];
            }
    }
}

/* ---- slots to their pixels: binning ----
 * Per slot the tree needs the smallest pixel and the number of pixels.  One pair of atomics per run of pixels went at
 * 22 G/s (2.5 of 3.6 ms on the 8192^2 u16 image, two thirds of the runs a slot of their own); a store to a random slot
 * runs four times as fast, LDS faster still.  So the runs are binned: slots of one branch follow each other, and
 * branches are numbered tile by tile, so the pixels of a tile fall into a few dozen bins of 4096 slots.
 *   k_bs_assign   one block per tile: every pixel's slot; the tile's items (slot, smallest pixel, pixels: its runs, or,
 *                 HASH, its distinct slots from a table in LDS) go to the tile's part of ent, bin by bin, and each
 *                 (tile, bin) with items gets a descriptor.  Items of a tile with more bins than its part of dsc holds
 *                 (one per eight pixels) go to the end of its part and are sent with atomics at the end (k_bs_rest)
 *   k_bs_desc     the descriptors sorted by bin (counts, a scan, places)
 *   k_bs_bin      one block per bin (or per part of a bin with many items): its items collected in LDS, its slots
 *                 written once */
#define BS_BIN 12
#define BS_BINS (1 << BS_BIN)
#define BS_BTAB 512      /* a tile's bins */
#define BS_PART 16384u   /* items of a part of a bin */
#define BS_PARTD 1024u   /* descriptors of a part (a constant image has one item a tile: 8192^2 1.9 ms in one part, 0.13 in 16) */

struct BsBins {
    uint2 *ent;      /* items: pixel, slot in bin | pixels << BS_BIN */
    uint2 *dsc;      /* per tile: bin, first item | items << 16 */
    uint2 *tile;     /* per tile: descriptors, items at the end of its part */
    uint32_t *slot;  /* every pixel's slot */
};

/* what k_bs_assign does with a tile's items: runs into bins, distinct slots into bins, or distinct slots sent with atomics
 * (small images: a dozen launches less, and a few hundred tiles wait little for each other; 1024^2 u8 0.73 against 0.76 ms,
 * 256x320 0.45 against 0.53, where the 8192^2 one takes 8.2 ms with bins and 11.5 with atomics) */
enum { BS_RUNS, BS_SLOTS, BS_SEND };

/* SPARSE: the branches are known (lab) and may be sparse; otherwise all are dense.
 * BS_SEND: first, cnt start cleared; nothing is done for more than cap slots (total[0]) */
template <bool D3, bool SPARSE, int KIND>
__global__ __launch_bounds__(256, KIND == BS_RUNS ? 6 : 8) void k_bs_assign(ImgView iv, BsGeo g, const uint4 *__restrict__ rec, const uint32_t *lab, BsSlots table,
                                                   BsBins o, uint32_t *__restrict__ first, uint32_t *__restrict__ cnt,
                                                   const unsigned long long *__restrict__ total, uint64_t cap)
{
    constexpr bool HASH = KIND != BS_RUNS;
    if (KIND == BS_SEND && *total > cap) return;
    auto send = [&](uint32_t s, uint32_t len, uint32_t p) {
        if (__hip_atomic_load(&first[s], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) > p) atomicMin(&first[s], p);
        atomicAdd(&cnt[s], len);
    };
    constexpr int ITEMS = HASH ? BS_TAB / 256 : 16; /* items a thread places */
    __shared__ uint32_t key[HASH ? BS_TAB : 1], num[HASH ? BS_TAB : 1], low[HASH ? BS_TAB : 1];
    constexpr int BT = KIND == BS_SEND ? 1 : BS_BTAB;
    __shared__ uint32_t bkey[BT], bcnt[BT], boff[BT], bidx[BT];
    __shared__ uint32_t nbin, nrest, wsum[4];
    const int tid = threadIdx.x;
    const BsTile t = bs_tile<BsShape3<D3>::TX, BsShape3<D3>::TY, BsShape3<D3>::TZ>(g, blockIdx.x);
    uint32_t before;
    const uint32_t px = bs_tile_pixels<D3>(t, before);
    const uint32_t d0 = before >> 3, dcap = ((before + px) >> 3) - d0;
    if constexpr (HASH)
        for (int i = tid; i < BS_TAB; i += 256) {
            key[i] = BS_NONE;
            num[i] = 0;
            low[i] = BS_NONE;
        }
    if constexpr (KIND != BS_SEND)
        for (int i = tid; i < BS_BTAB; i += 256) {
            bkey[i] = BS_NONE;
            bcnt[i] = 0;
        }
    if (tid == 0) nbin = nrest = 0;
    __syncthreads();
    /* an item without a bin: to the end of the tile's part */
    auto rest = [&](uint32_t p, uint32_t len) { o.ent[before + px - 1 - atomicAdd(&nrest, 1u)] = make_uint2(p, len << BS_BIN); };
    /* the table entry of a slot's bin, -1 when the table is crowded */
    auto bin_of = [&](uint32_t s) -> int {
        const uint32_t v = s >> BS_BIN;
        uint32_t h = (v * 2654435761u) >> 23;
        for (int i = 0; i < 16; i++) {
            const uint32_t k = atomicCAS(&bkey[h], BS_NONE, v);
            if (k == BS_NONE) bidx[h] = atomicAdd(&nbin, 1u);
            if (k == BS_NONE || k == v) return (int)h;
            h = (h + 1) & (BS_BTAB - 1);
        }
        return -1;
    };
    /* an item: its slot (BS_NONE: none), and table entry | place in the bin << 9 | (a run's pixels - 1) << 21 */
    uint32_t is[ITEMS], ir[ITEMS];
#pragma unroll
    for (int i0 = 0; i0 < 16; i0 += BS_AHEAD) {
        int p[BS_AHEAD];
        uint32_t v[BS_AHEAD], x[BS_AHEAD], s[BS_AHEAD];
        uint4 r[BS_AHEAD];
#pragma unroll
        for (int j = 0; j < BS_AHEAD; j++) {
            p[j] = bs_at<D3>(t, tid + 256 * (i0 + j));
            v[j] = p[j] >= 0 ? bs_key(iv, p[j]) : 0u;
        }
        if constexpr (SPARSE) {
#pragma unroll
            for (int j = 0; j < BS_AHEAD; j++) x[j] = p[j] >= 0 ? lab[p[j]] & ~BS_PEAK : 0u;
#pragma unroll
            for (int j = 0; j < BS_AHEAD; j++) r[j] = rec[x[j]];
#pragma unroll
            for (int j = 0; j < BS_AHEAD; j++) s[j] = p[j] >= 0 ? bs_slot(r[j], x[j], v[j], table) : BS_NONE;
        } else {
            bs_branches(rec, lab, p, v, x, r);
#pragma unroll
            for (int j = 0; j < BS_AHEAD; j++) s[j] = p[j] >= 0 ? r[j].z - v[j] : BS_NONE;
        }
#pragma unroll
        for (int j = 0; j < BS_AHEAD; j++) {
            const bool valid = p[j] >= 0;
            if (valid) o.slot[p[j]] = s[j];
            bool head;
            uint32_t len;
            int at;
            bs_runs(valid, s[j], false, head, len, at);
            if constexpr (HASH) {
                if (!head) continue;
                const int h = bs_find(key, s[j]);
                if (h < 0) {
                    if constexpr (KIND == BS_SEND) send(s[j], len, (uint32_t)p[j]);
                    else rest((uint32_t)p[j], len);
                } else {
                    atomicAdd(&num[h], len);
                    atomicMin(&low[h], (uint32_t)p[j]);
                }
            } else {
                const int k = i0 + j;
                is[k] = head ? s[j] : BS_NONE;
                ir[k] = 0;
                if (!head) continue;
                const int h = bin_of(s[j]);
                if (h < 0) {
                    rest((uint32_t)p[j], len);
                    is[k] = BS_NONE;
                } else ir[k] = (uint32_t)h | (atomicAdd(&bcnt[h], 1u) << 9) | ((len - 1u) << 21);
            }
        }
    }
    __syncthreads();
    if constexpr (KIND == BS_SEND) {
        for (int i = tid; i < BS_TAB; i += 256)
            if (key[i] != BS_NONE) send(key[i], num[i], low[i]);
        return;
    }
    if constexpr (HASH) {
#pragma unroll
        for (int k = 0; k < ITEMS; k++) {
            const int i = tid + 256 * k;
            is[k] = key[i];
            ir[k] = 0;
            if (is[k] == BS_NONE) continue;
            const int h = bin_of(is[k]);
            if (h < 0) {
                rest(low[i], num[i]);
                is[k] = BS_NONE;
            } else ir[k] = (uint32_t)h | (atomicAdd(&bcnt[h], 1u) << 9);
        }
        __syncthreads();
    }
    /* the bins' first items: prefix over the table (two entries a thread; bins beyond the descriptors hold none) */
    {
        const uint32_t b0 = 2u * tid, c0 = bkey[b0] != BS_NONE && bidx[b0] < dcap ? bcnt[b0] : 0u;
        const uint32_t c1 = bkey[b0 + 1] != BS_NONE && bidx[b0 + 1] < dcap ? bcnt[b0 + 1] : 0u;
        uint32_t pre = c0 + c1;
        const int lane = tid & 63;
#pragma unroll
        for (int of = 1; of < 64; of <<= 1) {
            const uint32_t u = __shfl_up(pre, of, 64);
            if (lane >= of) pre += u;
        }
        if (lane == 63) wsum[tid >> 6] = pre;
        __syncthreads();
        for (int w = 0; w < (tid >> 6); w++) pre += wsum[w];
        boff[b0] = pre - c0 - c1;
        boff[b0 + 1] = pre - c1;
    }
    __syncthreads();
    const int again = bs_opaque(tid);
#pragma unroll
    for (int k = 0; k < ITEMS; k++) {
        if (is[k] == BS_NONE) continue;
        const uint32_t h = ir[k] & (BS_BTAB - 1);
        uint32_t p, len;
        if constexpr (HASH) {
            p = low[tid + 256 * k];
            len = num[tid + 256 * k];
        } else {
            p = (uint32_t)bs_at<D3>(t, again + 256 * k);
            len = (ir[k] >> 21) + 1u;
        }
        if (bidx[h] >= dcap) rest(p, len);
        else o.ent[before + boff[h] + ((ir[k] >> 9) & 0xFFFu)] = make_uint2(p, (is[k] & (BS_BINS - 1)) | (len << BS_BIN));
    }
    for (int h = tid; h < BS_BTAB; h += 256)
        if (bkey[h] != BS_NONE && bidx[h] < dcap) o.dsc[d0 + bidx[h]] = make_uint2(bkey[h], boff[h] | (bcnt[h] << 16));
    __syncthreads();
    if (tid == 0) o.tile[blockIdx.x] = make_uint2(min(nbin, dcap), nrest);
}

/* descriptors of BS_DTILES tiles a block: their bins counted (bd: descriptors, be: items; one atomic per bin and block),
 * each one's place among its bin's */
#define BS_DTILES 16
template <bool D3>
__global__ __launch_bounds__(256) void k_bs_desc_count(BsGeo g, BsBins o, uint32_t *__restrict__ place, uint32_t *__restrict__ bd,
                                                       uint32_t *__restrict__ be, int tiles)
{
    __shared__ uint32_t key[BS_TAB], num[BS_TAB], items[BS_TAB];
    for (int i = threadIdx.x; i < BS_TAB; i += 256) {
        key[i] = BS_NONE;
        num[i] = 0;
        items[i] = 0;
    }
    __syncthreads();
    const int t0 = blockIdx.x * BS_DTILES, t1 = min(t0 + BS_DTILES, tiles);
    for (int pass = 0; pass < 2; pass++) {
        for (int ti = t0; ti < t1; ti++) {
            const BsTile t = bs_tile<BsShape3<D3>::TX, BsShape3<D3>::TY, BsShape3<D3>::TZ>(g, ti);
            uint32_t before;
            (void)bs_tile_pixels<D3>(t, before);
            const uint32_t nd = o.tile[ti].x;
            for (uint32_t d = threadIdx.x; d < nd; d += 256) {
                const uint32_t at = (before >> 3) + d;
                const uint2 q = o.dsc[at];
                if (pass == 0) {
                    const int h = bs_find(key, q.x);
                    if (h < 0) {
                        place[at] = 0x80000000u | atomicAdd(&bd[q.x], 1u);
                        atomicAdd(&be[q.x], q.y >> 16);
                    } else {
                        /* table entry and place in it; below 2^31: 2^11 entries, 2^13 descriptors */
                        place[at] = ((uint32_t)h << 16) | atomicAdd(&num[h], 1u);
                        atomicAdd(&items[h], q.y >> 16);
                    }
                } else {
                    const uint32_t v = place[at];
                    place[at] = (v & 0x80000000u) ? v & 0x7FFFFFFFu : num[v >> 16] + (v & 0xFFFFu);
                }
            }
        }
        __syncthreads();
        if (pass == 0) {
            for (int i = threadIdx.x; i < BS_TAB; i += 256)
                if (key[i] != BS_NONE) {
                    num[i] = atomicAdd(&bd[key[i]], num[i]);
                    atomicAdd(&be[key[i]], items[i]);
                }
            __syncthreads();
        }
    }
}

/* the descriptors in the order of their bins: first item, items */
template <bool D3>
__global__ __launch_bounds__(256) void k_bs_desc_place(BsGeo g, BsBins o, const uint32_t *__restrict__ place,
                                                       const uint32_t *__restrict__ bbase, uint2 *__restrict__ sorted)
{
    const BsTile t = bs_tile<BsShape3<D3>::TX, BsShape3<D3>::TY, BsShape3<D3>::TZ>(g, blockIdx.x);
    uint32_t before;
    (void)bs_tile_pixels<D3>(t, before);
    const uint32_t nd = o.tile[blockIdx.x].x;
    for (uint32_t d = threadIdx.x; d < nd; d += blockDim.x) {
        const uint32_t at = (before >> 3) + d;
        const uint2 q = o.dsc[at];
        sorted[bbase[q.x] + place[at]] = make_uint2(before + (q.y & 0xFFFFu), q.y >> 16);
    }
}

/* parts of every bin (entry NB: 0) */
__global__ __launch_bounds__(256) void k_bs_bin_parts(const uint32_t *__restrict__ bd, const uint32_t *__restrict__ be,
                                                      uint32_t *__restrict__ np, uint32_t NB)
{
    const uint32_t b = blockIdx.x * 256u + threadIdx.x;
    if (b > NB) return;
    if (b == NB) {
        np[b] = 0;
        return;
    }
    const uint32_t k = max((be[b] + BS_PART - 1) / BS_PART, (bd[b] + BS_PARTD - 1) / BS_PARTD);
    np[b] = max(1u, min(bd[b], k));
}

/* part -> bin; the slots of the bins with several parts cleared (their parts add with atomics) */
__global__ __launch_bounds__(256) void k_bs_bin_map(const uint32_t *__restrict__ pbase, uint32_t *__restrict__ pbin,
                                                    uint32_t *__restrict__ first, uint32_t *__restrict__ cnt, int64_t S)
{
    const uint32_t b = blockIdx.x, p0 = pbase[b], p1 = pbase[b + 1];
    for (uint32_t i = p0 + threadIdx.x; i < p1; i += 256) pbin[i] = b;
    if (p1 - p0 == 1) return;
    for (int i = threadIdx.x; i < BS_BINS; i += 256) {
        const int64_t s = ((int64_t)b << BS_BIN) + i;
        if (s < S) {
            first[s] = BS_NONE;
            cnt[s] = 0;
        }
    }
}

__global__ __launch_bounds__(256) void k_bs_bin(const uint2 *__restrict__ ent, const uint2 *__restrict__ sorted,
                                                const uint32_t *__restrict__ bbase, const uint32_t *__restrict__ pbase,
                                                const uint32_t *__restrict__ pbin, uint32_t NB, uint32_t *__restrict__ first,
                                                uint32_t *__restrict__ cnt, int64_t S)
{
    __shared__ uint32_t f[BS_BINS], c[BS_BINS];
    if (blockIdx.x >= pbase[NB]) return;
    const uint32_t b = pbin[blockIdx.x];
    const uint32_t np = pbase[b + 1] - pbase[b], part = blockIdx.x - pbase[b];
    const uint32_t nd = bbase[b + 1] - bbase[b];
    const uint32_t d0 = bbase[b] + (uint32_t)((uint64_t)nd * part / np), d1 = bbase[b] + (uint32_t)((uint64_t)nd * (part + 1) / np);
    for (int i = threadIdx.x; i < BS_BINS; i += 256) {
        f[i] = BS_NONE;
        c[i] = 0;
    }
    __syncthreads();
    const uint32_t lane = threadIdx.x & 63u, w = threadIdx.x >> 6;
    auto take = [&](uint2 e) {
        const uint32_t s = e.y & (BS_BINS - 1);
        atomicMin(&f[s], e.x);
        atomicAdd(&c[s], e.y >> BS_BIN);
    };
    /* a wave takes 64 descriptors at a time, four of them side by side */
    for (uint32_t d = d0 + 64u * w; d < d1; d += 256u) {
        const uint2 mine = d + lane < d1 ? sorted[d + lane] : make_uint2(0, 0);
        const uint32_t m = min(64u, d1 - d);
        for (uint32_t j = 0; j < m; j += 4) {
            uint32_t at[4], n[4], most = 0;
#pragma unroll
            for (int k = 0; k < 4; k++) {
                at[k] = __shfl(mine.x, (int)((j + k) & 63u), 64);
                n[k] = __shfl(mine.y, (int)((j + k) & 63u), 64);
                if (j + k >= m) n[k] = 0;
                most = max(most, n[k]);
            }
            for (uint32_t q = lane; q < most; q += 64u) {
                uint2 e[4];
#pragma unroll
                for (int k = 0; k < 4; k++)
                    if (q < n[k]) e[k] = ent[at[k] + q];
#pragma unroll
                for (int k = 0; k < 4; k++)
                    if (q < n[k]) take(e[k]);
            }
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < BS_BINS; i += 256) {
        const int64_t s = ((int64_t)b << BS_BIN) + i;
        if (s >= S) break;
        if (np == 1) {
            first[s] = f[i];
            cnt[s] = c[i];
        } else if (c[i]) {
            atomicMin(&first[s], f[i]);
            atomicAdd(&cnt[s], c[i]);
        }
    }
}

/* the items at the ends of the tiles' parts */
template <bool D3>
__global__ __launch_bounds__(64) void k_bs_rest(BsGeo g, BsBins o, uint32_t *__restrict__ first, uint32_t *__restrict__ cnt)
{
    const uint32_t n = o.tile[blockIdx.x].y;
    if (!n) return;
    const BsTile t = bs_tile<BsShape3<D3>::TX, BsShape3<D3>::TY, BsShape3<D3>::TZ>(g, blockIdx.x);
    uint32_t before;
    const uint32_t px = bs_tile_pixels<D3>(t, before);
    for (uint32_t i = threadIdx.x; i < n; i += 64) {
        const uint2 e = o.ent[before + px - 1 - i];
        const uint32_t s = o.slot[e.x];
        atomicMin(&first[s], e.x);
        atomicAdd(&cnt[s], e.y >> BS_BIN);
    }
}

/* ---- sparse branches (noise of many greys: a few pixels over thousands of keys) ---- */
/* every pixel's branch (lab) and its place among the branch's pixels (idx); the branches' pixel counts.  With pofs: the
 * same for the pixels of the branches in pieces, and their pieces */
template <bool D3, bool PIECE>
__global__ __launch_bounds__(256) void k_bs_count(ImgView iv, BsGeo g, const uint4 *__restrict__ rec, uint32_t *lab,
                                                  uint32_t *__restrict__ idx, uint32_t *__restrict__ bcnt,
                                                  const uint32_t *__restrict__ pval, const uint32_t *__restrict__ pofs, int piece)
{
    __shared__ uint32_t key[BS_TAB], num[BS_TAB];
    const BsTile t = bs_tile<BsShape3<D3>::TX, BsShape3<D3>::TY, BsShape3<D3>::TZ>(g, blockIdx.x);
    for (int i = threadIdx.x; i < BS_TAB; i += 256) {
        key[i] = BS_NONE;
        num[i] = 0;
    }
    __syncthreads();
    constexpr uint32_t DIRECT = 0x80000000u; /* placed in memory: idx is already there */
    uint32_t place[16];                       /* table entry << 16 | place among the tile's pixels of the branch */
#pragma unroll
    for (int i0 = 0; i0 < 16; i0 += BS_AHEAD) {
        int p[BS_AHEAD];
        uint32_t v[BS_AHEAD], x[BS_AHEAD];
        uint4 r[BS_AHEAD];
#pragma unroll
        for (int j = 0; j < BS_AHEAD; j++) {
            p[j] = bs_at<D3>(t, (int)threadIdx.x + 256 * (i0 + j));
            v[j] = p[j] >= 0 ? bs_key(iv, p[j]) : 0u;
        }
        if constexpr (!PIECE) bs_branches(rec, lab, p, v, x, r);
#pragma unroll
        for (int j = 0; j < BS_AHEAD; j++) {
            bool valid = p[j] >= 0;
            if constexpr (PIECE) {
                if (valid) {
                    const uint32_t b = lab[p[j]] & ~BS_PEAK;
                    valid = pofs[b + 1] > pofs[b];
                    x[j] = pofs[b] + ((pval[b] - v[j]) >> piece);
                }
            } else if (valid) __hip_atomic_store(&lab[p[j]], BS_PEAK | x[j], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            bool head;
            uint32_t len, b = 0;
            int at;
            bs_runs(valid, x[j], false, head, len, at);
            if (head) {
                const int h = bs_find(key, x[j]);
                b = h < 0 ? DIRECT | atomicAdd(&bcnt[x[j]], len) : ((uint32_t)h << 16) | atomicAdd(&num[h], len);
            }
            b = __shfl(b, at, 64) + (uint32_t)((int)(threadIdx.x & 63) - at);
            if (valid && (b & DIRECT)) idx[p[j]] = b & ~DIRECT;
            place[i0 + j] = valid ? b : DIRECT;
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < BS_TAB; i += 256)
        if (key[i] != BS_NONE) num[i] = atomicAdd(&bcnt[key[i]], num[i]);
    __syncthreads();
    const int again = bs_opaque((int)threadIdx.x);
#pragma unroll
    for (int i = 0; i < 16; i++)
        if (!(place[i] & DIRECT)) {
            const int p = bs_at<D3>(t, again + 256 * i);
            idx[p] = num[place[i] >> 16] + (place[i] & 0xFFFFu);
        }
}

/* the keys of the sparse branches and pieces, each one's together */
__global__ __launch_bounds__(256) void k_bs_scatter(ImgView iv, const uint4 *__restrict__ rec, const uint32_t *__restrict__ lab,
                                                    const uint32_t *__restrict__ idx, BsSlots table, uint32_t *__restrict__ skey,
                                                    int64_t n)
{
    const int64_t p = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (p >= n) return;
    const uint32_t x = lab[p] & ~BS_PEAK;
    const uint4 r = rec[x];
    if (!r.w) return;
    const uint32_t v = bs_key(iv, p);
    uint32_t z = r.z;
    if (r.w == BS_PIECES) {
        const uint2 q = table.prec[z + ((table.pval[x] - v) >> table.piece)];
        if (!q.y) return;
        z = q.x;
    }
    skey[z + idx[p]] = v;
}

/* the m keys k (a power of two) sorted from the highest down by threads threads, this one number i0; sync between them */
template <class F> __device__ __forceinline__ void bs_bitonic(uint32_t *k, int m, int i0, int threads, F sync)
{
    for (int a = 2; a <= m; a <<= 1)
        for (int h = a >> 1; h > 0; h >>= 1) {
            for (int i = i0; i < m / 2; i += threads) {
                const int lo = ((i & -h) << 1) | (i & (h - 1)), hi = lo + h;
                const uint32_t u = k[lo], v = k[hi];
                if ((u < v) == ((lo & a) == 0)) {
                    k[lo] = v;
                    k[hi] = u;
                }
            }
            sync();
        }
}

#define BS_ST 1024
/* The keys of the runs of slots listed in mid, each sorted from the highest down (bitonic): up to 64 keys by a wave in
 * registers, up to 512 by a wave in its part of the LDS, more by the block.  Most runs are short (8192^2
 * u16 noise: 1.56 ms when a block and its barriers took one at a time). */
__global__ __launch_bounds__(BS_ST) void k_bs_sort(const uint2 *__restrict__ mid, const uint32_t *__restrict__ nmid,
                                                 uint32_t *__restrict__ skey)
{
    constexpr uint32_t WAVES = BS_ST / 64, PART = BS_SORT / WAVES;
    __shared__ uint32_t k[BS_SORT];
    const uint32_t N = *nmid;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    for (uint32_t j = blockIdx.x * WAVES + w; j < N; j += gridDim.x * WAVES) {
        const uint2 r = mid[j];
        if (r.y > PART) continue;
        if (r.y <= 64u) {
            uint32_t u = lane < (int)r.y ? skey[r.x + lane] : 0u;
            for (int a = 2; a <= 64; a <<= 1)
                for (int h = a >> 1; h > 0; h >>= 1) {
                    const uint32_t v = __shfl_xor(u, h, 64);
                    /* the lower lane of a pair keeps the higher key where its run of a keys falls */
                    u = ((lane & a) == 0) == ((lane & h) == 0) ? max(u, v) : min(u, v);
                }
            if (lane < (int)r.y) skey[r.x + lane] = u;
            continue;
        }
        uint32_t *q = k + w * PART;
        int m = 128;
        while (m < (int)r.y) m <<= 1;
        auto sync = []() {
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        };
        for (int i = lane; i < m; i += 64) q[i] = i < (int)r.y ? skey[r.x + i] : 0u;
        sync();
        bs_bitonic(q, m, lane, 64, sync);
        for (int i = lane; i < (int)r.y; i += 64) skey[r.x + i] = q[i];
        sync();
    }
    __syncthreads();
    for (uint32_t j = blockIdx.x; j < N; j += gridDim.x) {
        const uint2 r = mid[j];
        if (r.y <= PART) continue;
        int m = 2 * (int)PART;
        while (m < (int)r.y) m <<= 1;
        for (int i = threadIdx.x; i < m; i += BS_ST) k[i] = i < (int)r.y ? skey[r.x + i] : 0u;
        __syncthreads();
        bs_bitonic(k, m, (int)threadIdx.x, BS_ST, []() { __syncthreads(); });
        for (int i = threadIdx.x; i < (int)r.y; i += BS_ST) skey[r.x + i] = k[i];
        __syncthreads();
    }
}

/* ------------------------------------------------------------------------------------------------ */
/* nodes                                                                                            */
/* ------------------------------------------------------------------------------------------------ */
/* the nodes along the branches, BT * 16 slots a block: levelroot pixel, own pixels, parent (the next node;
 * k_bs_link sets the last ones of the branches); nid = the nodes before every slot, before = the pixels of the nodes
 * before every node (and one past the last), nodes[0] their number.  Nothing is done for more than cap slots.  (BT: see BS_BIG) */
template <int BT>
__global__ __launch_bounds__(BT) void k_bs_nodes(const uint32_t *__restrict__ first, const uint32_t *__restrict__ cnt, BsChain ch,
                                                  uint32_t *__restrict__ nid, uint32_t *__restrict__ npix,
                                                  uint32_t *__restrict__ area, uint32_t *__restrict__ before,
                                                  int32_t *__restrict__ cpar, uint32_t *__restrict__ head,
                                                  unsigned long long *__restrict__ nodes, const unsigned long long *__restrict__ total,
                                                  uint64_t cap)
{
    typedef unsigned long long u64;
    constexpr int ROWS = 16, TILE = BT * ROWS, WAVES = BT / 64;
    __shared__ u64 wsum[WAVES], carry;
    const int64_t S = (int64_t)*total;
    if ((uint64_t)S > cap) return;
    const uint32_t t = bs_tile_ticket(ch);
    if ((int64_t)t * TILE > S) return;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int64_t s0 = (int64_t)t * TILE + w * (64 * ROWS) + lane;
    uint32_t p[ROWS], a[ROWS];
    u64 mine = 0, sum;
#pragma unroll
    for (int i = 0; i < ROWS; i++) {
        const int64_t s = s0 + 64 * i;
        p[i] = s < S ? first[s] : BS_NONE;
        a[i] = p[i] != BS_NONE ? cnt[s] : 0u;
    }
    /* nodes << 31 | pixels: both below 2^31 in all */
#pragma unroll
    for (int i = 0; i < ROWS; i++) mine += (p[i] != BS_NONE ? 1ull << 31 : 0ull) + a[i];
    (void)bs_wave_prefix(mine, sum);
    if (lane == 0) wsum[w] = sum;
    __syncthreads();
    u64 all = 0;
    for (int k = 0; k < WAVES; k++) all += wsum[k];
    if (w == 0) {
        const u64 b = bs_look_back(ch, t, all);
        if (threadIdx.x == 0) carry = b;
    }
    __syncthreads();
    u64 base = carry;
    for (int k = 0; k < w; k++) base += wsum[k];
#pragma unroll
    for (int i = 0; i < ROWS; i++) {
        const int64_t s = s0 + 64 * i;
        const u64 v = (p[i] != BS_NONE ? 1ull << 31 : 0ull) + a[i];
        const u64 at = base + bs_wave_prefix(v, sum);
        base += sum;
        const uint32_t c = (uint32_t)(at >> 31);
        if (s <= S) nid[s] = c;
        if (s == S) {
            before[c] = (uint32_t)(at & 0x7FFFFFFFull);
            *nodes = c;
        }
        if (p[i] == BS_NONE) continue;
        npix[c] = p[i];
        area[c] = a[i];
        before[c] = (uint32_t)(at & 0x7FFFFFFFull);
        cpar[c] = (int32_t)c + 1;
        head[c] = 0;
    }
}

struct BsLink {
    uint32_t n0, n1; /* the branch's nodes */
    int32_t at;      /* the node it hangs below, -1 for a root */
    uint32_t into;   /* the branch of that node, BS_NONE when that is a root's */
};

__global__ __launch_bounds__(256) void k_bs_link(const uint4 *__restrict__ rec, const uint32_t *__restrict__ base,
                                                 const uint32_t *__restrict__ nid, BsSlots table, int32_t *__restrict__ cpar,
                                                 BsLink *__restrict__ link, uint32_t *__restrict__ nch, uint32_t *__restrict__ head,
                                                 uint32_t *__restrict__ tarea, uint32_t G)
{
    const uint32_t x = blockIdx.x * 256u + threadIdx.x;
    if (x >= G) return;
    tarea[x] = 0;
    BsLink k;
    k.n0 = nid[base[x]];
    k.n1 = nid[base[x + 1]];
    k.at = -1;
    k.into = BS_NONE;
    if (k.n1 > k.n0) {
        const uint4 r = rec[x];
        if ((int32_t)r.x >= 0) {
            uint4 ry;
            k.into = bs_climb(rec, r.y, r.x, ry);
            k.at = (int32_t)nid[bs_slot(ry, k.into, r.x, table)];
            if ((int32_t)ry.x >= 0) atomicAdd(&nch[k.into], 1u);
            else k.into = BS_NONE; /* a root's total is not needed */
        }
        cpar[k.n1 - 1] = k.at;
        head[k.n0] = k.n0; /* its running maximum: the first node of every node's branch */
    }
    link[x] = k;
}

/* ------------------------------------------------------------------------------------------------ */
/* attribute records                                                                                */
/* ------------------------------------------------------------------------------------------------ */
template <int G> struct BsShape {
    static constexpr int NS = G == 2 ? 3 : (G == 3 ? 4 : (G == 4 ? 9 : 0));
    static constexpr bool EXT = G == 1;
};

/* sums (or extents) of the pixels of every node (A.area: their number).  A tile collects them in coordinates of its own (below 64, or 16 in
 * 3D), in which the moments of all its 4096 pixels fit packed words: pixels and first moments in one (16 + 3 x 16 bits
 * in 3D, 16 + 2 x 24 in 2D), squares in one, products in one; a run of pixels of one row adds closed-form sums.  The
 * tile's origin (and the node's grey, which all its pixels share) enters when an item is sent. */
/* threads of a block: the table takes up to 57 KB of LDS, two blocks a CU */
#define BS_OWN(G) ((G) == 1 || (G) == 4 ? 1024 : 512)
template <int G, bool D3>
__global__ __launch_bounds__(BS_OWN(G)) void k_bs_own(ImgView iv, BsGeo g, int ox, int oy, int oz, const uint32_t *__restrict__ slot,
                                                const uint32_t *__restrict__ nid, DevAttr A)
{
    constexpr int BT = BS_OWN(G);
    constexpr int TX = BsShape3<D3>::TX, TY = BsShape3<D3>::TY, TZ = BsShape3<D3>::TZ;
    constexpr int NQ = G == 1 ? 1 : (G == 4 ? 3 : 1); /* packed words per item */
    constexpr int B1 = D3 ? 16 : 24, B2 = D3 ? 21 : 32;
    __shared__ uint32_t key[BS_TAB];
    __shared__ unsigned long long q[G == 1 ? 1 : NQ * BS_TAB];
    __shared__ uint32_t ext[G == 1 ? 6 * BS_TAB : 1];
    __shared__ uint32_t grey[G == 3 ? BS_TAB : 1];
    const BsTile t = bs_tile<TX, TY, TZ>(g, blockIdx.x);
    for (int i = threadIdx.x; i < BS_TAB; i += BT) {
        key[i] = BS_NONE;
        if constexpr (G == 1)
            for (int k = 0; k < 6; k++) ext[k * BS_TAB + i] = k < 3 ? BS_NONE : 0u;
        else
            for (int k = 0; k < NQ; k++) q[k * BS_TAB + i] = 0ull;
    }
    __syncthreads();
    const int64_t X = t.x0 + ox, Y = t.y0 + oy, Z = t.z0 + oz;
    /* an item's sums from its packed words to its record */
    auto send = [&](uint32_t c, unsigned long long q0, unsigned long long q1, unsigned long long q2, uint32_t v) {
        const unsigned long long m1 = (1ull << B1) - 1, m2 = (1ull << B2) - 1;
        const int64_t n = (int64_t)(q0 & 0xFFFF);
        const int64_t sx = (int64_t)((q0 >> 16) & m1), sy = (int64_t)((q0 >> (16 + B1)) & m1), sz = D3 ? (int64_t)(q0 >> 48) : 0;
        int64_t s[9] = { n * X + sx, n * Y + sy, n * Z + sz, 0, 0, 0, 0, 0, 0 };
        if constexpr (G == 3) {
            s[3] = s[2] * v; s[2] = s[1] * v; s[1] = s[0] * v; s[0] = n * (int64_t)v;
        }
        if constexpr (G == 4) {
            const int64_t xx = (int64_t)(q1 & m2), yy = (int64_t)((q1 >> B2) & m2), zz = D3 ? (int64_t)(q1 >> (2 * B2)) : 0;
            const int64_t xy = (int64_t)(q2 & m2), yz = D3 ? (int64_t)((q2 >> B2) & m2) : 0, xz = D3 ? (int64_t)(q2 >> (2 * B2)) : 0;
            s[3] = n * X * X + 2 * X * sx + xx;
            s[4] = n * Y * Y + 2 * Y * sy + yy;
            s[5] = n * Z * Z + 2 * Z * sz + zz;
            s[6] = n * X * Y + X * sy + Y * sx + xy;
            s[7] = n * Y * Z + Y * sz + Z * sy + yz;
            s[8] = n * X * Z + X * sz + Z * sx + xz;
        }
        /* an item that is the whole node (as most are in a noisy image) is stored: an atomic costs four stores */
        if (n == (int64_t)A.area[c]) {
#pragma unroll
            for (int i = 0; i < BsShape<G>::NS; i++)
                if (s[i]) A.s[i][c] = s[i];
            return;
        }
#pragma unroll
        for (int i = 0; i < BsShape<G>::NS; i++)
            if (s[i]) atomicAdd((unsigned long long *)&A.s[i][c], (unsigned long long)s[i]);
    };
    auto send_ext = [&](uint32_t c, const uint32_t (&e)[6]) {
        const uint32_t o[3] = { (uint32_t)X, (uint32_t)Y, (uint32_t)Z };
#pragma unroll
        for (int k = 0; k < 3; k++) {
            atomicMin(&A.mn[k][c], o[k] + e[k]);
            atomicMax(&A.mx[k][c], o[k] + e[3 + k]);
        }
    };
    uint32_t node[BS_AHEAD];
    for (int i = 0; i < BS_TILE / BT; i++) {
        if (i % BS_AHEAD == 0) {
            /* the chains of BS_AHEAD pixels side by side */
#pragma unroll
            for (int j = 0; j < BS_AHEAD; j++) {
                const int p = bs_at<D3>(t, (int)threadIdx.x + BT * (i + j));
                node[j] = p >= 0 ? slot[p] : BS_NONE;
            }
#pragma unroll
            for (int j = 0; j < BS_AHEAD; j++)
                if (node[j] != BS_NONE) node[j] = nid[node[j]];
        }
        const int l = (int)threadIdx.x + BT * i;
        const uint32_t x = (uint32_t)(l % TX), y = (uint32_t)((l / TX) % TY), z = D3 ? (uint32_t)(l / (TX * TY)) : 0u;
        const int p = bs_at<D3>(t, l);
        uint32_t c = node[0];
#pragma unroll
        for (int j = 1; j < BS_AHEAD; j++) c = i % BS_AHEAD == j ? node[j] : c;
        bool head;
        uint32_t L;
        int at;
        bs_runs(p >= 0, c, x == 0, head, L, at);
        if (!head) continue;
        const int h = bs_find(key, c);
        if constexpr (G == 1) {
            const uint32_t e[6] = { x, y, z, x + L, y + 1, z + 1 };
            if (h < 0) send_ext(c, e);
            else {
#pragma unroll
                for (int k = 0; k < 3; k++) {
                    atomicMin(&ext[k * BS_TAB + h], e[k]);
                    atomicMax(&ext[(3 + k) * BS_TAB + h], e[3 + k]);
                }
            }
        } else {
            typedef unsigned long long u64;
            const u64 n = L, sx = (u64)L * x + (u64)L * (L - 1) / 2;
            const u64 q0 = n | (sx << 16) | ((n * y) << (16 + B1)) | (D3 ? (n * z) << 48 : 0ull);
            u64 q1 = 0, q2 = 0;
            if constexpr (G == 4) {
                const u64 xx = (u64)L * x * x + (u64)x * L * (L - 1) + (u64)(L - 1) * L * (2 * L - 1) / 6;
                q1 = xx | ((n * y * y) << B2) | (D3 ? (n * z * z) << (2 * B2) : 0ull);
                q2 = (sx * y) | (D3 ? ((n * y * z) << B2) | ((sx * z) << (2 * B2)) : 0ull);
            }
            const uint32_t v = G == 3 ? bs_key(iv, p) : 0u;
            if (h < 0) send(c, q0, q1, q2, v);
            else {
                atomicAdd(&q[h], q0);
                if constexpr (G == 4) {
                    atomicAdd(&q[BS_TAB + h], q1);
                    atomicAdd(&q[2 * BS_TAB + h], q2);
                }
                if constexpr (G == 3) grey[h] = v;
            }
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < BS_TAB; i += BT) {
        const uint32_t c = key[i];
        if (c == BS_NONE) continue;
        if constexpr (G == 1) {
            uint32_t e[6];
#pragma unroll
            for (int k = 0; k < 6; k++) e[k] = ext[k * BS_TAB + i];
            send_ext(c, e);
        } else {
            send(c, q[i], G == 4 ? q[(NQ - 2) * BS_TAB + i] : 0ull, G == 4 ? q[(NQ - 1) * BS_TAB + i] : 0ull, G == 3 ? grey[i] : 0u);
        }
    }
}

/* (branch's first node, value) as one key: its running maximum along the nodes is the maximum inside the branch */
struct BsRun {
    const uint32_t *cbase, *v;
    uint32_t flip; /* BS_NONE: minima as maxima of the complement */
    __host__ __device__ uint64_t operator()(uint32_t c) const { return ((uint64_t)cbase[c] << 32) | (v[c] ^ flip); }
};

/* prefixes over the nodes: exclusive sums of the counts and sums (one entry past the end), running maxima of the
 * extents */
struct BsPrefix {
    const uint32_t *area;
    const int64_t *s[DCF_MAX_SUMS];
    const uint64_t *mn[3], *mx[3];
};

/* per branch, filled from its children */
struct BsTotals {
    uint32_t *done; /* children that have arrived */
    DevAttr T;
};

/* Branch totals from the leaves up: a branch adds its total to its parent branch (B.T; a root's total is not needed),
 * and the last child to arrive goes on with the parent.  Nobody waits.  B.T ends with every branch's total from its
 * children; its own nodes' come from E. */
template <int G>
__global__ __launch_bounds__(256) void k_bs_totals(const BsLink *__restrict__ link, const uint32_t *__restrict__ nch, BsPrefix E,
                                                   BsTotals B, uint32_t nb)
{
    constexpr int NS = BsShape<G>::NS;
    uint32_t x = blockIdx.x * 256u + threadIdx.x;
    if (x >= nb || nch[x]) return;
    for (;;) {
        const BsLink k = link[x];
        const uint32_t y = k.into;
        if (y == BS_NONE) return; /* below a root, a root, or a branch without pixels */
        atomicAdd(&B.T.area[y], E.area[k.n1] - E.area[k.n0] + bs_lda(&B.T.area[x]));
#pragma unroll
        for (int i = 0; i < NS; i++) {
            if (!E.s[i]) continue; /* all zero */
            const unsigned long long v =
                (unsigned long long)(E.s[i][k.n1] - E.s[i][k.n0]) + (unsigned long long)bs_lda(&B.T.s[i][x]);
            if (v) atomicAdd((unsigned long long *)&B.T.s[i][y], v);
        }
        if constexpr (BsShape<G>::EXT)
            for (int i = 0; i < 3; i++) {
                atomicMin(&B.T.mn[i][y], min(~(uint32_t)E.mn[i][k.n1 - 1], bs_lda(&B.T.mn[i][x])));
                atomicMax(&B.T.mx[i][y], max((uint32_t)E.mx[i][k.n1 - 1], bs_lda(&B.T.mx[i][x])));
            }
        /* only atomics pass between the threads, all of them device-scope (B.T and done must stay so: a plain access here would
         * race): waiting for them to be performed is all of a release that atomics past the L2 need on this GPU, and orders
         * them before the count.  A fence would also write back and drop the caches, once per branch (22 ms instead of 0.8 for a
         * batch tree of 128 images) */
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        if (atomicAdd(&B.done[y], 1u) + 1 != nch[y]) return;
        x = y;
    }
}

/* every branch's total into the own records A of the node it hangs below.  The background's nodes take hundreds of
 * thousands of branches: a block collects BS_JOIN of them in a table first */
#define BS_JOIN 2048
template <int G>
__global__ __launch_bounds__(256) void k_bs_join(const BsLink *__restrict__ link, BsPrefix E, BsTotals B, DevAttr A, uint32_t nb)
{
    constexpr int NS = BsShape<G>::NS;
    constexpr bool EXT = BsShape<G>::EXT;
    constexpr int TAB = 512;
    __shared__ uint32_t key[TAB], area[TAB];
    __shared__ unsigned long long sum[NS > 0 ? NS * TAB : 1];
    __shared__ uint32_t ext[EXT ? 6 * TAB : 1];
    for (int i = threadIdx.x; i < TAB; i += 256) {
        key[i] = BS_NONE;
        area[i] = 0;
        for (int k = 0; k < NS; k++) sum[k * TAB + i] = 0ull;
        if constexpr (EXT)
            for (int k = 0; k < 6; k++) ext[k * TAB + i] = k < 3 ? BS_NONE : 0u;
    }
    __syncthreads();
    for (uint32_t j = threadIdx.x; j < BS_JOIN; j += 256) {
        const uint32_t x = blockIdx.x * BS_JOIN + j;
        if (x >= nb) break;
        const BsLink k = link[x];
        if (k.at < 0) continue;
        const uint32_t c = (uint32_t)k.at;
        int h = -1;
        uint32_t at = (c * 2654435761u) >> 23;
        for (int i = 0; i < 4 && h < 0; i++) {
            const uint32_t o = atomicCAS(&key[at], BS_NONE, c);
            if (o == BS_NONE || o == c) h = (int)at;
            at = (at + 1) & (TAB - 1);
        }
        const uint32_t ar = E.area[k.n1] - E.area[k.n0] + B.T.area[x];
        atomicAdd(h < 0 ? &A.area[c] : &area[h], ar);
#pragma unroll
        for (int i = 0; i < NS; i++) {
            if (!E.s[i]) continue; /* all zero */
            const unsigned long long v = (unsigned long long)(E.s[i][k.n1] - E.s[i][k.n0]) + (unsigned long long)B.T.s[i][x];
            if (v) {
                if (h < 0) atomicAdd((unsigned long long *)&A.s[i][c], v);
                else atomicAdd(&sum[i * TAB + h], v);
            }
        }
        if constexpr (EXT)
            for (int i = 0; i < 3; i++) {
                const uint32_t lo = min(~(uint32_t)E.mn[i][k.n1 - 1], B.T.mn[i][x]), hi = max((uint32_t)E.mx[i][k.n1 - 1], B.T.mx[i][x]);
                atomicMin(h < 0 ? &A.mn[i][c] : &ext[i * TAB + h], lo);
                atomicMax(h < 0 ? &A.mx[i][c] : &ext[(3 + i) * TAB + h], hi);
            }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < TAB; i += 256) {
        const uint32_t c = key[i];
        if (c == BS_NONE) continue;
        atomicAdd(&A.area[c], area[i]);
#pragma unroll
        for (int k = 0; k < NS; k++)
            if (sum[k * TAB + i]) atomicAdd((unsigned long long *)&A.s[k][c], sum[k * TAB + i]);
        if constexpr (EXT)
            for (int k = 0; k < 3; k++) {
                atomicMin(&A.mn[k][c], ext[k * TAB + i]);
                atomicMax(&A.mx[k][c], ext[(3 + k) * TAB + i]);
            }
    }
}

/* ------------------------------------------------------------------------------------------------ */
/* results                                                                                          */
/* ------------------------------------------------------------------------------------------------ */
/* Blocks of the kernels that go through an array in order (BsChain): BS_BIG threads for a large image, 256 for a small
 * one.  A ticket is an atomic on one word (about 25 ns each) and a look-back passes the words of all blocks in flight,
 * so a large image wants few and large tiles; a small one wants a block on every CU. */
#define BS_BIG 1024

/* the levelroots as a bitmap with the levelroots before every word (rk: 64 pixels a word, bits in x, y, levelroots before
 * it in z), the other pixels' parents; a block takes BT * 16 pixels */
template <int BT>
__global__ __launch_bounds__(BT) void k_bs_parent(const uint32_t *__restrict__ slot, const uint32_t *__restrict__ first,
                                                  int32_t *__restrict__ parent, uint4 *__restrict__ rk, BsChain ch, int64_t n)
{
    constexpr int WORDS = BT / 4, PER = WORDS / 64; /* words of a block, of a lane of its first wave */
    __shared__ uint64_t word[WORDS];
    const uint32_t t = bs_tile_ticket(ch);
    const int64_t p0 = (int64_t)t * (BT * 16);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    for (int i0 = 0; i0 < 16; i0 += 4) {
        uint32_t s[4], r[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int64_t p = p0 + (w * 16 + i0 + j) * 64 + lane;
            s[j] = p < n ? slot[p] : 0u;
        }
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int64_t p = p0 + (w * 16 + i0 + j) * 64 + lane;
            r[j] = p < n ? first[s[j]] : BS_NONE;
        }
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int64_t p = p0 + (w * 16 + i0 + j) * 64 + lane;
            const bool root = p < n && r[j] == (uint32_t)p;
            if (p < n && !root) parent[p] = (int32_t)r[j];
            const uint64_t m = __ballot(root);
            if (lane == 0) word[w * 16 + i0 + j] = m;
        }
    }
    __syncthreads();
    if (w != 0) return;
    uint64_t m[PER];
    unsigned long long sum, mine = 0;
#pragma unroll
    for (int i = 0; i < PER; i++) {
        m[i] = word[lane * PER + i];
        mine += (unsigned long long)__popcll(m[i]);
    }
    unsigned long long pre = bs_wave_prefix(mine, sum);
    pre += bs_look_back(ch, t, sum);
#pragma unroll
    for (int i = 0; i < PER; i++) {
        if (p0 + (lane * PER + i) * 64 < n)
            rk[(p0 >> 6) + lane * PER + i] = make_uint4((uint32_t)m[i], (uint32_t)(m[i] >> 32), (uint32_t)pre, 0u);
        pre += (unsigned long long)__popcll(m[i]);
    }
}

/* raster number of levelroot r */
__device__ __forceinline__ uint32_t bs_rank(const uint4 *__restrict__ rk, uint32_t r)
{
    const uint4 v = rk[r >> 6];
    const uint64_t bits = ((uint64_t)v.y << 32) | v.x;
    return v.z + (uint32_t)__popcll(bits & ((1ull << (r & 63)) - 1));
}

/* areas: the running sum of the nodes' own pixels (and the totals that k_bs_join added) that starts anew with every
 * branch: crec[c] = (the parent's levelroot or BS_NONE, area).  A thread takes four nodes.  cidx: the node of every raster
 * number, when those are known (p2n).
 * The nodes lie along the branches here and in raster order in the results; records of eight bytes are written here in
 * order and gathered there, since a scattered store of four bytes costs about four times as much as a gather. */
template <int BT>
__global__ __launch_bounds__(BT) void k_bs_area(const uint32_t *__restrict__ own, const uint32_t *__restrict__ head,
                                                const uint32_t *__restrict__ npix, const int32_t *__restrict__ cpar, BsChain ch,
                                                uint2 *__restrict__ crec, const uint32_t *__restrict__ p2n,
                                                uint32_t *__restrict__ cidx, int64_t K)
{
    constexpr int WAVES = BT / 64;
    __shared__ uint32_t wsum[WAVES], carry;
    __shared__ int wstart[WAVES];
    const uint32_t t = bs_tile_ticket(ch);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int64_t c0 = (int64_t)t * (BT * 4) + threadIdx.x * 4;
    uint32_t v[4], rq[4];
    bool h[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int64_t c = c0 + i;
        v[i] = c < K ? own[c] : 0u;
        h[i] = c < K && (c == 0 || head[c] != 0);
        const int32_t q = c < K ? cpar[c] : -1;
        rq[i] = q < 0 ? BS_NONE : npix[q];
        if (cidx && c < K) cidx[p2n[npix[c]]] = (uint32_t)c;
    }
    /* sums since the thread's last start, and whether it has one */
    uint32_t run = 0;
    bool any = false;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        run = h[i] ? v[i] : run + v[i];
        any = any || h[i];
    }
    /* segmented inclusive prefix over the wave */
    uint32_t x = run;
    bool f = any;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t y = __shfl_up(x, o, 64);
        const int g = __shfl_up((int)f, o, 64);
        if (lane >= o && !f) {
            x += y;
            f = g != 0;
        }
    }
    if (lane == 63) {
        wsum[w] = x;
        wstart[w] = f;
    }
    /* before this thread, inside the wave */
    uint32_t pre = __shfl_up(x, 1, 64);
    bool closed = __shfl_up((int)f, 1, 64) != 0;
    if (lane == 0) {
        pre = 0;
        closed = false;
    }
    __syncthreads();
    if (w == 0) {
        uint32_t all = 0;
        bool whole = false;
        for (int i = 0; i < WAVES; i++) {
            all = wstart[i] ? wsum[i] : all + wsum[i];
            whole = whole || wstart[i];
        }
        const unsigned long long b = bs_look_back(ch, t, all, whole);
        if (threadIdx.x == 0) carry = (uint32_t)b;
    }
    __syncthreads();
    uint32_t in = carry;
    for (int i = 0; i < w; i++) in = wstart[i] ? wsum[i] : in + wsum[i];
    uint32_t s = closed ? pre : in + pre;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        s = h[i] ? v[i] : s + v[i];
        if (c0 + i < K) crec[c0 + i] = make_uint2(rq[i], s);
    }
}

/* the results in raster order: every pixel's node, and the levelroots' parents and node arrays (cidx: their nodes' places
 * along the branches).  Bound by the gathers: 0.70 ms for 67 million pixels and 15 million nodes (8192^2 u16), 0.58 for 134
 * million of a 512^3 u8 volume; with k_bs_area's records in place of scattered stores one 8192^2 tree went from 8.2 to 7.6. */
__global__ __launch_bounds__(256) void k_bs_result(ImgView iv, const uint32_t *__restrict__ slot, const uint32_t *__restrict__ nid,
                                                   const uint2 *__restrict__ crec, const uint4 *__restrict__ rk,
                                                   int32_t *__restrict__ parent, uint32_t *__restrict__ p2n, int32_t *__restrict__ npar,
                                                   float *__restrict__ ngrey, uint32_t *__restrict__ area, uint32_t *__restrict__ nroot,
                                                   uint32_t *__restrict__ cidx, int64_t n)
{
    /* four words of 64 pixels a wave, so that each lane has four chains of gathers under way */
    const int lane = threadIdx.x & 63;
    const int64_t w0 = ((int64_t)blockIdx.x * 4 + (threadIdx.x >> 6)) * 4;
    uint32_t r[4], k[4], c[4], nk[4];
    uint2 q[4];
    bool root[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int64_t p = (w0 + j) * 64 + lane;
        r[j] = p < n ? (uint32_t)parent[p] : 0u;
        root[j] = false;
        if (p < n) {
            const uint4 v = rk[p >> 6];
            root[j] = (((((uint64_t)v.y << 32) | v.x) >> lane) & 1ull) != 0;
        }
        if (root[j]) r[j] = (uint32_t)p; /* (its parent is not written yet) */
    }
#pragma unroll
    for (int j = 0; j < 4; j++) c[j] = root[j] ? slot[r[j]] : 0u;
#pragma unroll
    for (int j = 0; j < 4; j++) k[j] = bs_rank(rk, r[j]);
#pragma unroll
    for (int j = 0; j < 4; j++)
        if (root[j]) c[j] = nid[c[j]];
#pragma unroll
    for (int j = 0; j < 4; j++) q[j] = root[j] ? crec[c[j]] : make_uint2(BS_NONE, 0u);
#pragma unroll
    for (int j = 0; j < 4; j++) nk[j] = q[j].x != BS_NONE ? bs_rank(rk, q[j].x) : BS_NONE;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int64_t p = (w0 + j) * 64 + lane;
        if (p < n) p2n[p] = k[j];
        if (!root[j]) continue;
        parent[p] = (int32_t)q[j].x;
        npar[k[j]] = (int32_t)nk[j];
        ngrey[k[j]] = bs_grey(iv, p);
        area[k[j]] = q[j].y;
        if (nroot) nroot[k[j]] = (uint32_t)p;
        if (cidx) cidx[k[j]] = c[j];
    }
}

/* records in raster order (the areas too where k_bs_result did not run) */
template <int G>
__global__ __launch_bounds__(256) void k_bs_records(const uint32_t *__restrict__ cidx, const uint32_t *__restrict__ cbase,
                                                    const uint2 *__restrict__ crec, BsPrefix E, DevAttr A, int64_t K)
{
    const int64_t k = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (k >= K) return;
    const uint32_t c = cidx[k];
    if (crec) A.area[k] = crec[c].y;
    if constexpr (G > 0) {
        const uint32_t b = cbase[c];
#pragma unroll
        for (int i = 0; i < BsShape<G>::NS; i++) A.s[i][k] = E.s[i] ? E.s[i][c + 1] - E.s[i][b] : 0;
        if constexpr (BsShape<G>::EXT)
            for (int i = 0; i < 3; i++) {
                A.mn[i][k] = ~(uint32_t)E.mn[i][c];
                A.mx[i][k] = (uint32_t)E.mx[i][c];
            }
    }
}

/* a[0 .. total) = v, b[0 .. total) = w; nothing for more than cap */
__global__ __launch_bounds__(256) void k_bs_fill2(uint32_t *__restrict__ a, uint32_t v, uint32_t *__restrict__ b, uint32_t w,
                                                  const unsigned long long *__restrict__ total, uint64_t cap)
{
    const uint64_t n = *total;
    if (n > cap) return;
    for (uint64_t i = ((uint64_t)blockIdx.x * 256u + threadIdx.x) * 4u; i < n; i += (uint64_t)gridDim.x * 1024u) {
        if (i + 4 <= n) {
            *(uint4 *)(a + i) = make_uint4(v, v, v, v);
            *(uint4 *)(b + i) = make_uint4(w, w, w, w);
        } else
            for (uint64_t j = i; j < n; j++) {
                a[j] = v;
                b[j] = w;
            }
    }
}

__global__ __launch_bounds__(256) void k_bs_fill32(uint32_t *__restrict__ a, uint32_t v, int64_t n)
{
    const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
    if (i + 4 <= n) *(uint4 *)(a + i) = make_uint4(v, v, v, v);
    else
        for (int64_t j = i; j < n; j++) a[j] = v;
}

/* ------------------------------------------------------------------------------------------------ */
/* host side                                                                                        */
/* ------------------------------------------------------------------------------------------------ */
static inline unsigned nblk(int64_t n, int bs) { return (unsigned)((n + bs - 1) / bs); }

namespace {
struct Scratch {
    dcf_ctx *ctx;
    std::vector<void *> ptrs;
    template <class T> T *get(size_t count)
    {
        void *p = dcf_alloc(ctx, count * sizeof(T));
        if (p) ptrs.push_back(p);
        return (T *)p;
    }
    /* gives one block back before the others */
    void drop(void *p)
    {
        auto it = std::find(ptrs.begin(), ptrs.end(), p);
        if (it == ptrs.end()) return;
        ptrs.erase(it);
        dcf_release(ctx, p);
    }
    ~Scratch()
    {
        for (void *p : ptrs) dcf_release(ctx, p);
    }
};
}

static int fill(dcf_ctx *ctx, void *a, uint32_t v, int64_t words)
{
    DCF_LAUNCH(ctx, "k_bs_fill", k_bs_fill32, dim3(nblk(words, 1024)), dim3(256), 0, (uint32_t *)a, v, words);
    return DCF_OK;
}

#define BS_TRY(call)                \
    do {                            \
        const int rc_ = (call);     \
        if (rc_ != DCF_OK) return rc_; \
    } while (0)

/* a hipcub device algorithm: sized, given scratch, run */
#define BS_CUB(...)                                                                          \
    do {                                                                                     \
        size_t need_ = 0;                                                                    \
        auto run_ = [&](void *tmp_, size_t &sz_) -> hipError_t { return __VA_ARGS__; };      \
        DCF_HIP(ctx, run_(nullptr, need_));                                                  \
        void *t_ = sc.get<char>(need_ ? need_ : 16);                                         \
        if (!t_) return dcf_set_error(ctx, DCF_ENOMEM, "scan scratch");                      \
        DCF_HIP(ctx, run_(t_, need_));                                                       \
        sc.drop(t_);                                                                         \
    } while (0)

typedef hipcub::CountingInputIterator<uint32_t> BsIota;

/* ---- exclusive prefixes of several sums at once ----
 * Sums of tiles, their prefixes (one block per sum), the prefixes inside the tiles: three launches for a group instead of
 * two for each of its up to nine sums, twice per build (4096^2 shape filter 7.84 -> 7.52 ms, 203x187x151 volume 1.22 -> 1.11). */
#define BS_SUM 4096
struct BsSums {
    const int64_t *in[DCF_MAX_SUMS];
    int64_t *out[DCF_MAX_SUMS];
};

/* the 16 elements of sum i that a thread holds: wave w of the block takes 1024 in a row, 64 at a time */
__device__ __forceinline__ void bs_sum_load(const int64_t *__restrict__ in, int64_t n, unsigned long long (&v)[16])
{
    const int64_t c0 = (int64_t)blockIdx.x * BS_SUM + (threadIdx.x >> 6) * 1024 + (threadIdx.x & 63);
#pragma unroll
    for (int j = 0; j < 16; j++) v[j] = c0 + 64 * j < n ? (unsigned long long)in[c0 + 64 * j] : 0ull;
}

__global__ __launch_bounds__(256) void k_bs_sum_tiles(BsSums a, unsigned long long *__restrict__ part, int64_t n)
{
    __shared__ unsigned long long wsum[4];
    unsigned long long v[16], s = 0, sum;
    bs_sum_load(a.in[blockIdx.y], n, v);
#pragma unroll
    for (int j = 0; j < 16; j++) s += v[j];
    (void)bs_wave_prefix(s, sum);
    if ((threadIdx.x & 63) == 0) wsum[threadIdx.x >> 6] = sum;
    __syncthreads();
    if (threadIdx.x == 0) part[(int64_t)blockIdx.y * gridDim.x + blockIdx.x] = wsum[0] + wsum[1] + wsum[2] + wsum[3];
}

__global__ __launch_bounds__(1024) void k_bs_sum_top(unsigned long long *__restrict__ part, int64_t tiles)
{
    __shared__ unsigned long long wsum[16];
    unsigned long long *p = part + (int64_t)blockIdx.x * tiles, carry = 0;
    const int w = threadIdx.x >> 6;
    for (int64_t t0 = 0; t0 < tiles; t0 += 1024) {
        const int64_t t = t0 + threadIdx.x;
        unsigned long long sum, pre = bs_wave_prefix(t < tiles ? p[t] : 0ull, sum);
        if ((threadIdx.x & 63) == 0) wsum[w] = sum;
        __syncthreads();
        unsigned long long all = 0;
        for (int k = 0; k < 16; k++) {
            if (k < w) pre += wsum[k];
            all += wsum[k];
        }
        if (t < tiles) p[t] = carry + pre;
        carry += all;
        __syncthreads();
    }
}

__global__ __launch_bounds__(256) void k_bs_sum_out(BsSums a, const unsigned long long *__restrict__ part, int64_t n)
{
    __shared__ unsigned long long wsum[4];
    unsigned long long v[16], s = 0, sum;
    bs_sum_load(a.in[blockIdx.y], n, v);
#pragma unroll
    for (int j = 0; j < 16; j++) s += v[j];
    (void)bs_wave_prefix(s, sum);
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) wsum[w] = sum;
    __syncthreads();
    unsigned long long base = part[(int64_t)blockIdx.y * gridDim.x + blockIdx.x];
    for (int k = 0; k < w; k++) base += wsum[k];
    int64_t *out = a.out[blockIdx.y];
    const int64_t c0 = (int64_t)blockIdx.x * BS_SUM + w * 1024 + (threadIdx.x & 63);
#pragma unroll
    for (int j = 0; j < 16; j++) {
        const unsigned long long pre = base + bs_wave_prefix(v[j], sum);
        if (c0 + 64 * j < n) out[c0 + 64 * j] = (int64_t)pre;
        base += sum;
    }
}

/* exclusive sums / running maxima of the nodes' records A but the areas (K entries, the sums' arrays K + 1) */
static int prefixes(dcf_ctx *ctx, Scratch &sc, const DevAttr &A, const uint32_t *cbase, int64_t *const *Es, uint64_t *const *Emn,
                    uint64_t *const *Emx, int64_t K)
{
    BsSums a = {};
    int sums = 0;
    for (int i = 0; i < A.nsum; i++)
        if (Es[i]) {
            a.in[sums] = A.s[i];
            a.out[sums++] = Es[i];
        }
    if (sums) {
        const unsigned tiles = nblk(K + 1, BS_SUM);
        unsigned long long *part = sc.get<unsigned long long>((size_t)tiles * sums);
        if (!part) return dcf_set_error(ctx, DCF_ENOMEM, "prefix sums");
        DCF_LAUNCH(ctx, "k_bs_sums", k_bs_sum_tiles, dim3(tiles, (unsigned)sums), dim3(256), 0, a, part, K + 1);
        DCF_LAUNCH(ctx, "k_bs_sums", k_bs_sum_top, dim3((unsigned)sums), dim3(1024), 0, part, (int64_t)tiles);
        DCF_LAUNCH(ctx, "k_bs_sums", k_bs_sum_out, dim3(tiles, (unsigned)sums), dim3(256), 0, a, (const unsigned long long *)part, K + 1);
        sc.drop(part);
    }
    for (int i = 0; A.has_ext && i < 3; i++)
        for (int hi = 0; hi < 2; hi++) {
            const BsRun op{ cbase, hi ? A.mx[i] : A.mn[i], hi ? 0u : BS_NONE };
            hipcub::TransformInputIterator<uint64_t, BsRun, BsIota> in(BsIota(0u), op);
            BS_CUB(hipcub::DeviceScan::InclusiveScan(tmp_, sz_, in, hi ? Emx[i] : Emn[i], hipcub::Max(), (int)K, ctx->stream));
        }
    return DCF_OK;
}

/* the sums of z of a flat image (one slice, at z = 0) are zero: they have no arrays, and no passes (four of group 4's nine) */
static bool zero_sum(int grp, bool flat, int i)
{
    return flat && ((grp == 2 && i == 2) || (grp == 3 && i == 3) || (grp == 4 && (i == 2 || i == 5 || i == 7 || i == 8)));
}

/* records of n nodes (or branches) for group grp beside their areas, one spare entry; neutral values */
static int records(dcf_ctx *ctx, Scratch &sc, DevAttr &a, int grp, bool flat, int64_t n)
{
    a.nsum = grp == 2 ? 3 : (grp == 3 ? 4 : (grp == 4 ? 9 : 0));
    a.has_ext = grp == 1;
    for (int i = 0; i < a.nsum; i++) {
        if (zero_sum(grp, flat, i)) continue;
        if (!(a.s[i] = sc.get<int64_t>((size_t)n + 1))) return dcf_set_error(ctx, DCF_ENOMEM, "attribute records");
        BS_TRY(fill(ctx, a.s[i], 0u, 2 * (n + 1)));
    }
    for (int i = 0; a.has_ext && i < 3; i++) {
        a.mn[i] = sc.get<uint32_t>((size_t)n + 1);
        a.mx[i] = sc.get<uint32_t>((size_t)n + 1);
        if (!a.mn[i] || !a.mx[i]) return dcf_set_error(ctx, DCF_ENOMEM, "attribute records");
        BS_TRY(fill(ctx, a.mn[i], BS_NONE, n + 1));
        BS_TRY(fill(ctx, a.mx[i], 0u, n + 1));
    }
    return DCF_OK;
}

/* one attempt with room for ecap saddle edges: *edges = 0 when they had room, else their number, and nothing is changed */
static int basin_build(dcf_tree *t, int grp, bool nodes, uint64_t ecap, uint64_t *edges)
{
    dcf_ctx *ctx = t->ctx;
    const int64_t n = t->n;
    *edges = 0;
    /* node slots stay below 2^31 */
    if (n >= ((int64_t)1 << 30)) return dcf_set_error(ctx, DCF_EUNSUPPORTED, "images are limited to 2^30 pixels");
    const int is3d = t->bimg ? t->batch3d : t->dims[2] > 1;
    const int mode = is3d ? (t->conn == 26 ? 3 : 2) : (t->conn == 8 ? 1 : 0);
    Scratch sc{ ctx, {} };
    ImgView px;
    px.img = t->img;
    px.dtype = t->dtype;
    px.invert = t->tree_min;
    px.gmax = t->gmax;
    ImgView iv = px;
    if (t->dtype == DCF_F32) {
        uint32_t *rank = sc.get<uint32_t>((size_t)n), maxr = 0;
        if (!rank) return dcf_set_error(ctx, DCF_ENOMEM, "grey ranks");
        BS_TRY(dcf_rank_keys(t, rank, &maxr));
        iv.img = rank;
        iv.dtype = DCF_KEY32;
        iv.invert = 0;
        iv.gmax = nullptr;
    }
    BsGeo g;
    g.W = (int)t->dims[0];
    g.H = (int)t->dims[1];
    g.D = (int)t->dims[2];
    g.n = n;
    g.bimg = t->bimg;
    g.nbatch = t->nbatch;
    const int tx = is3d ? 16 : 64;
    g.ntx = (g.W + tx - 1) / tx;
    g.nty = (g.H + tx - 1) / tx;
    const int64_t tiles = t->bimg ? t->basin_tiles : (int64_t)g.ntx * g.nty * (is3d ? (g.D + tx - 1) / tx : 1);

    /* ---- basins and saddles ---- */
    /* A small image is bound by launches and waits: its arrays are made for as many peaks, edges and dense slots as there
     * may be, so that the host reads no count back before the number of nodes (256x320 u8: 0.45 -> 0.24 ms with the scans
     * inside their kernels).  Ranks of a float image are mostly sparse.  The line, with the one between atomics and bins below
     * (builds as a small and as a large image): 1024^2 u8 disks 0.51 and 0.53 ms, u8 noise 0.84 and 0.85; 1448^2 u16 value noise 0.54
     * and 0.62; 2048^2 0.73 and 0.78, but u8 disks 1.02 and 0.83; 2880^2 u8 disks 1.81 and 1.28; 160^3 0.64 and 0.60, 256^3 1.68 and
     * 1.18. */
    const bool few = n <= ((int64_t)1 << 22) && iv.dtype != DCF_KEY32;
    const uint64_t dense_cap = (uint64_t)(2 * n + (1 << 20));
    const bool big = n > ((int64_t)1 << 22);
    uint32_t *lab = sc.get<uint32_t>((size_t)n);
    uint32_t *pval = sc.get<uint32_t>((size_t)n + 1);
    uint2 *raw = sc.get<uint2>((size_t)ecap);
    /* counters: [0] peaks, [1] saddle edges, [2] slots, [3] nodes, then per Boruvka round the edges and components left,
     * flags, tickets; then the state words of the prefixes: slots, nodes (of a dense and of a sparse attempt), levelroots,
     * areas.  All start at zero. */
    const size_t zslots = (size_t)n / 1024 + 2, znodes = (size_t)(dense_cap >> BS_BIN) + 2, zsparse = (size_t)(8 * n / BS_BINS) + 300,
                 zroots = (size_t)n / 4096 + 2, zarea = (size_t)n / 1024 + 2;
    const size_t zall = 128 + zslots + znodes + zsparse + zroots + zarea;
    unsigned long long *count = sc.get<unsigned long long>(zall);
    if (!lab || !pval || !count || !raw) return dcf_set_error(ctx, DCF_ENOMEM, "basin arrays");
    uint32_t *ecount = (uint32_t *)(count + 8), *rcount = (uint32_t *)(count + 40), *more = (uint32_t *)(count + 72),
             *nmid = (uint32_t *)(count + 80), *ticket = (uint32_t *)(count + 96);
    unsigned long long *z = count + 128;
    const BsChain ch_slots{ z, ticket }, ch_nodes{ z + zslots, ticket + 1 }, ch_sparse{ z + zslots + znodes, ticket + 2 },
        ch_roots{ z + zslots + znodes + zsparse, ticket + 3 }, ch_area{ z + zslots + znodes + zsparse + zroots, ticket + 4 };
    BS_TRY(fill(ctx, count, 0u, (int64_t)zall * 2));
    BsBor b = {};
    b.count = count;
    b.ecount = ecount;
    b.deep = ecount + 32;
    b.rcount = rcount;
    b.pval = pval;
    uint32_t *base = nullptr, *nch = nullptr, *done = nullptr;
    /* the arrays of the forest and of the branches, for G peaks and E edges */
    auto forest = [&](uint64_t G, uint64_t E) -> bool {
        b.rec = sc.get<uint4>((size_t)G + 1);
        b.hook = sc.get<uint32_t>((size_t)G + 1);
        b.comp = sc.get<uint32_t>((size_t)G + 1);
        base = sc.get<uint32_t>((size_t)G + 1);
        nch = sc.get<uint32_t>((size_t)G + 1);
        done = sc.get<uint32_t>((size_t)G + 1);
        bool ok = b.rec && b.hook && b.comp && base && nch && done;
        for (int i = 0; i < 2; i++) {
            b.e[i].w = sc.get<uint64_t>((size_t)E);
            b.e[i].ab = sc.get<uint2>((size_t)E);
            b.best[i] = sc.get<uint64_t>((size_t)G + 1);
            b.roots[i] = sc.get<uint32_t>((size_t)G + 1);
            ok = ok && b.e[i].w && b.e[i].ab && b.best[i] && b.roots[i];
        }
        return ok;
    };
    const dim3 pg(nblk(n, 256)), tg((unsigned)tiles), bl(256);
    uint64_t G = (uint64_t)n, E = ecap; /* at most */
    if (few && !forest(G, E)) return dcf_set_error(ctx, DCF_ENOMEM, "basin graph");
#define BS_ASCENT(M)                                                                                                       \
    {                                                                                                                      \
        DCF_LAUNCH(ctx, "k_bs_ascent", k_bs_ascent<M>, tg, bl, 0, iv, g, lab, pval, raw, ecap, count);                     \
        for (int r = 0; r < (few ? 1 : 3); r++)                                                                            \
            DCF_LAUNCH(ctx, "k_bs_border", k_bs_border<M>, tg, bl, 0, g, lab, more, r, b, few ? 1 : 0);                    \
        break;                                                                                                             \
    }
    switch (mode) {
    case 0: BS_ASCENT(0);
    case 1: BS_ASCENT(1);
    case 2: BS_ASCENT(2);
    default: BS_ASCENT(3);
    }
    unsigned long long host[4] = {};
    if (!few) {
        DCF_HIP(ctx, hipMemcpyAsync(host, count, 16, hipMemcpyDeviceToHost, ctx->stream));
        DCF_HIP(ctx, hipStreamSynchronize(ctx->stream));
        if (host[1] > ecap) {
            *edges = host[1];
            return DCF_OK;
        }
        G = host[0];
        E = host[1];
        if (!forest(G, E)) return dcf_set_error(ctx, DCF_ENOMEM, "basin graph");
        const dim3 ig(std::min(std::max(nblk((int64_t)G, 256), 1024u), 65536u));
        if (is3d) DCF_LAUNCH(ctx, "k_bs_init", k_bs_init<true>, ig, bl, 0, g, lab, (const uint32_t *)more + 2, (int)tiles, b);
        else DCF_LAUNCH(ctx, "k_bs_init", k_bs_init<false>, ig, bl, 0, g, lab, (const uint32_t *)more + 2, (int)tiles, b);
    }

    /* ---- spanning forest ---- */
    if (E) {
        const dim3 eg(std::max(1u, std::min(nblk((int64_t)(few ? E / 4 : E), 256), 4096u)));
        if (!few)
            DCF_LAUNCH(ctx, "k_bs_edges", k_bs_edges, eg, bl, 0, iv, (const uint32_t *)lab, (const uint2 *)raw, b, ecap);
        else if (is3d)
            DCF_LAUNCH(ctx, "k_bs_edges", k_bs_edges_far<true>, eg, bl, 0, iv, g, lab, (const uint32_t *)more, (int)tiles, (const uint2 *)raw, b, ecap);
        else
            DCF_LAUNCH(ctx, "k_bs_edges", k_bs_edges_far<false>, eg, bl, 0, iv, g, lab, (const uint32_t *)more, (int)tiles, (const uint2 *)raw, b, ecap);
        /* whole-GPU rounds until about a thousand components should be left (a round leaves between a fourth
         * and a seventh of them on the images measured; any number is right, the last block takes what is left);
         * an image has at most a peak for two pixels, noise one for five to ten (u8 noise of 2048^2, a round too few for G / 40:
         * 1.75 against 2.31 ms; G / 4 as fast, 1.72) */
        const uint64_t g0 = few ? G / 10 : G, e0 = few ? E / 5 : E;
        int rounds = 0;
        while (rounds < 30 && (g0 >> (2 * rounds)) > 1024u) rounds++;
        for (int r = 0; r < rounds; r++) {
            const unsigned eb = std::max(1u, std::min(nblk((int64_t)(e0 >> r), 256), 4096u));
            const unsigned rb = std::max(1u, std::min(nblk((int64_t)(g0 >> r), 256), 4096u));
            DCF_LAUNCH(ctx, "k_bs_hook", k_bs_hook, dim3(eb), bl, 0, b, r);
            DCF_LAUNCH(ctx, "k_bs_merge", k_bs_merge, dim3(rb), bl, 0, b, r);
            DCF_LAUNCH(ctx, "k_bs_contract", k_bs_contract, dim3(std::max(1u, nblk((int64_t)eb * 256, BS_CHUNK))), bl, 0, b, r);
        }
        DCF_HIP(ctx, hipFuncSetAttribute((const void *)k_bs_finish, hipFuncAttributeMaxDynamicSharedMemorySize, BS_FLDS));
        DCF_LAUNCH(ctx, "k_bs_finish", k_bs_finish, dim3(1), dim3(BS_FT), BS_FLDS, b, rounds);
    }
    sc.drop(raw);
    for (int i = 0; i < 2; i++) {
        sc.drop(b.e[i].w);
        sc.drop(b.e[i].ab);
        sc.drop(b.best[i]);
        sc.drop(b.roots[i]);
    }
    sc.drop(b.hook);
    sc.drop(b.comp);

    /* ---- slots ---- */
    uint32_t *slot = sc.get<uint32_t>((size_t)n);
    if (!slot) return dcf_set_error(ctx, DCF_ENOMEM, "slots");
    DCF_LAUNCH(ctx, "k_bs_slots", k_bs_slots, dim3(nblk((int64_t)G + 1, 1024)), bl, 0, b.rec, (const uint32_t *)pval, base,
               (const unsigned long long *)count, count + 2, ch_slots, nch, done);
    /* the nodes of S slots (at most): slot arrays, node arrays for at most Kc nodes */
    uint32_t *first = nullptr, *cnt = nullptr, *nid = nullptr, *npix = nullptr, *own = nullptr, *before = nullptr, *head = nullptr;
    int32_t *cpar = nullptr;
    auto slots = [&](uint64_t S) -> bool {
        const size_t Kc = (size_t)std::min<uint64_t>(S, (uint64_t)n) + 1;
        first = sc.get<uint32_t>((size_t)S + 1);
        cnt = sc.get<uint32_t>((size_t)S + 1);
        nid = sc.get<uint32_t>((size_t)S + 1);
        npix = sc.get<uint32_t>(Kc);
        own = sc.get<uint32_t>(Kc);
        before = sc.get<uint32_t>(Kc);
        head = sc.get<uint32_t>(Kc);
        cpar = sc.get<int32_t>(Kc);
        return first && cnt && nid && npix && own && before && head && cpar;
    };
    BsSlots table{ pval, nullptr, nullptr, BS_PIECE };
    BsBins bins{ nullptr, nullptr, nullptr, slot };
    const unsigned long long *total = count + 2;
#define BS_ASSIGN(SP, KIND, cap)                                                                                            \
    {                                                                                                                       \
        if (is3d)                                                                                                           \
            DCF_LAUNCH(ctx, "k_bs_assign", (k_bs_assign<true, SP, KIND>), tg, bl, 0, iv, g, (const uint4 *)b.rec, lab, table, bins, \
                       first, cnt, total, cap);                                                                             \
        else                                                                                                                \
            DCF_LAUNCH(ctx, "k_bs_assign", (k_bs_assign<false, SP, KIND>), tg, bl, 0, iv, g, (const uint4 *)b.rec, lab, table, bins, \
                       first, cnt, total, cap);                                                                             \
    }
    auto nodes_of = [&](uint64_t S, const BsChain &ch) -> int {
        if (big)
            DCF_LAUNCH(ctx, "k_bs_nodes", k_bs_nodes<BS_BIG>, dim3((unsigned)(S / (BS_BIG * 16)) + 1), dim3(BS_BIG), 0,
                       (const uint32_t *)first, (const uint32_t *)cnt, ch, nid, npix, own, before, cpar, head, count + 3, total, S);
        else
            DCF_LAUNCH(ctx, "k_bs_nodes", k_bs_nodes<256>, dim3((unsigned)(S / (256 * 16)) + 1), bl, 0, (const uint32_t *)first,
                       (const uint32_t *)cnt, ch, nid, npix, own, before, cpar, head, count + 3, total, S);
        return DCF_OK;
    };
    if (few) {
        if (!slots(dense_cap)) return dcf_set_error(ctx, DCF_ENOMEM, "slot arrays");
        DCF_LAUNCH(ctx, "k_bs_fill", k_bs_fill2, dim3(std::min(nblk((int64_t)dense_cap, 1024), 1024u)), bl, 0, first, BS_NONE, cnt, 0u,
                   total, dense_cap);
        BS_ASSIGN(false, BS_SEND, dense_cap);
        BS_TRY(nodes_of(dense_cap, ch_nodes));
    }
    DCF_HIP(ctx, hipMemcpyAsync(host, count, sizeof host, hipMemcpyDeviceToHost, ctx->stream));
    DCF_HIP(ctx, hipStreamSynchronize(ctx->stream));
    if (host[1] > ecap) {
        *edges = host[1];
        return DCF_OK;
    }
    G = host[0];
    unsigned long long S = host[2];
    /* one slot per key while that is at most two per pixel (or small); else by each branch's pixel count (with one or four per
     * pixel all images measured stay within 2 %) */
    const bool sparse = S > std::min<uint64_t>(dense_cap, 0x7FFFFFF0u);
    const uint32_t loose = (uint32_t)std::min<int64_t>(8, 0x7FFFFFF0 / n);
    const dim3 gg(nblk((int64_t)G + 1, 256));
    uint32_t *bcnt = nullptr, *skey = nullptr, *pofs = nullptr, *psum = nullptr, *pcnt = nullptr, NP = 0;
    uint2 *mid = nullptr, *prec = nullptr;
    if (sparse) {
        if (few)
            for (void *p : { (void *)first, (void *)cnt, (void *)nid, (void *)npix, (void *)own, (void *)before, (void *)head, (void *)cpar })
                sc.drop(p);
        bcnt = sc.get<uint32_t>((size_t)G);
        uint32_t *size = sc.get<uint32_t>((size_t)G + 1);
        if (!bcnt || !size) return dcf_set_error(ctx, DCF_ENOMEM, "branch counts");
        BS_TRY(fill(ctx, bcnt, 0u, (int64_t)G));
        BS_TRY(fill(ctx, count + 2, 0u, 2));
#define BS_COUNT(D3, PC, C) \
    DCF_LAUNCH(ctx, "k_bs_count", (k_bs_count<D3, PC>), tg, bl, 0, iv, g, (const uint4 *)b.rec, lab, slot, C, (const uint32_t *)pval, \
               (const uint32_t *)pofs, table.piece)
        if (is3d) BS_COUNT(true, false, bcnt);
        else BS_COUNT(false, false, bcnt);
        uint32_t *np = sc.get<uint32_t>((size_t)G + 1);
        pofs = sc.get<uint32_t>((size_t)G + 1);
        if (!np || !pofs) return dcf_set_error(ctx, DCF_ENOMEM, "branch pieces");
        const uint64_t most = (uint64_t)(n >> 6) + 4096; /* pieces */
        for (;;) {
            DCF_LAUNCH(ctx, "k_bs_range", k_bs_range, dim3(std::min(gg.x, 1024u)), bl, 0, (const uint4 *)b.rec, (const uint32_t *)pval,
                       (const uint32_t *)bcnt, size, np, loose, table.piece, (uint32_t)G, count + 2);
            unsigned long long sum[3]; /* slots, (nodes,) pieces */
            DCF_HIP(ctx, hipMemcpyAsync(sum, count + 2, sizeof sum, hipMemcpyDeviceToHost, ctx->stream));
            DCF_HIP(ctx, hipStreamSynchronize(ctx->stream));
            S = sum[0];
            NP = (uint32_t)sum[2];
            if (sum[2] <= most) break;
            /* (pieces of 2^24 keys: at most 65 for each of n / BS_SORT branches) */
            while (sum[2] > most) {
                sum[2] >>= 1;
                table.piece++;
            }
            BS_TRY(fill(ctx, count + 2, 0u, 2));
            BS_TRY(fill(ctx, count + 4, 0u, 2));
        }
        if (NP) {
            BS_CUB(hipcub::DeviceScan::ExclusiveSum(tmp_, sz_, np, pofs, (int)(G + 1), ctx->stream));
            pcnt = sc.get<uint32_t>((size_t)NP);
            psum = sc.get<uint32_t>((size_t)NP + 1);
            prec = sc.get<uint2>((size_t)NP);
            uint32_t *psize = sc.get<uint32_t>((size_t)NP + 1);
            if (!pcnt || !psum || !prec || !psize) return dcf_set_error(ctx, DCF_ENOMEM, "branch pieces");
            BS_TRY(fill(ctx, pcnt, 0u, NP));
            if (is3d) BS_COUNT(true, true, pcnt);
            else BS_COUNT(false, true, pcnt);
            DCF_LAUNCH(ctx, "k_bs_piece", k_bs_piece_size, dim3(nblk((int64_t)NP + 1, 256)), bl, 0, (const uint32_t *)pcnt, psize, NP, table.piece,
                       count + 2);
            DCF_HIP(ctx, hipMemcpyAsync(&S, count + 2, 8, hipMemcpyDeviceToHost, ctx->stream));
            DCF_HIP(ctx, hipStreamSynchronize(ctx->stream));
            if (S > 0x7FFFFFF0u) return dcf_set_error(ctx, DCF_EUNSUPPORTED, "too many grey values for branches of %d pixels", (int)BS_SORT);
            BS_CUB(hipcub::DeviceScan::ExclusiveSum(tmp_, sz_, psize, psum, (int)(NP + 1), ctx->stream));
            DCF_LAUNCH(ctx, "k_bs_piece", k_bs_piece_sum, gg, bl, 0, (const uint32_t *)pofs, (const uint32_t *)psum, size, (uint32_t)G);
        }
        sc.drop(np);
        BS_CUB(hipcub::DeviceScan::ExclusiveSum(tmp_, sz_, size, base, (int)(G + 1), ctx->stream));
        if (!(mid = sc.get<uint2>((size_t)G + NP))) return dcf_set_error(ctx, DCF_ENOMEM, "branch list");
        DCF_LAUNCH(ctx, "k_bs_base", k_bs_base, gg, bl, 0, b.rec, (const uint32_t *)pval, (const uint32_t *)bcnt, (const uint32_t *)base,
                   (const uint32_t *)pofs, loose, mid, nmid, (uint32_t)G);
        if (NP)
            DCF_LAUNCH(ctx, "k_bs_piece", k_bs_piece_base, dim3(nblk(NP, 256)), bl, 0, (const uint32_t *)pval, (const uint32_t *)pofs,
                       (const uint32_t *)psum, (const uint32_t *)pcnt, (const uint32_t *)base, prec, mid, nmid, table.piece, NP,
                       (uint32_t)G);
        if (!(skey = sc.get<uint32_t>((size_t)S))) return dcf_set_error(ctx, DCF_ENOMEM, "branch keys");
        table.skey = skey;
        table.prec = prec;
        DCF_LAUNCH(ctx, "k_bs_scatter", k_bs_scatter, pg, bl, 0, iv, (const uint4 *)b.rec, (const uint32_t *)lab, (const uint32_t *)slot,
                   table, skey, n);
        DCF_LAUNCH(ctx, "k_bs_sort", k_bs_sort, dim3(512), dim3(BS_ST), 0, (const uint2 *)mid, (const uint32_t *)nmid, skey);
    }
    if (!few || sparse) {
        if (!slots(S)) return dcf_set_error(ctx, DCF_ENOMEM, "slot arrays");
        if (n <= ((int64_t)1 << 22)) {
            DCF_LAUNCH(ctx, "k_bs_fill", k_bs_fill2, dim3(std::min(nblk((int64_t)S, 1024), 1024u)), bl, 0, first, BS_NONE, cnt, 0u, total,
                       (uint64_t)S);
            if (sparse) BS_ASSIGN(true, BS_SEND, (uint64_t)S)
            else BS_ASSIGN(false, BS_SEND, (uint64_t)S)
        } else {
            const uint32_t NB = (uint32_t)((S >> BS_BIN) + 1);
            uint32_t *bd = sc.get<uint32_t>(2 * (size_t)NB + 1), *be = bd ? bd + NB + 1 : nullptr, *bbase = sc.get<uint32_t>((size_t)NB + 1);
            uint32_t *np = sc.get<uint32_t>((size_t)NB + 1), *pbase = sc.get<uint32_t>((size_t)NB + 1);
            /* more than there can be (a bin has max(items / BS_PART, descriptors / BS_PARTD) + 1 at most) */
            const uint32_t parts = NB + (uint32_t)(n / BS_PART) + (uint32_t)((n >> 3) / BS_PARTD) + 1;
            uint32_t *pbin = sc.get<uint32_t>((size_t)parts);
            const size_t dn = (size_t)(n >> 3) + 1;
            bins.ent = sc.get<uint2>((size_t)n);
            bins.dsc = sc.get<uint2>(dn);
            bins.tile = sc.get<uint2>((size_t)tiles);
            uint32_t *place = sc.get<uint32_t>(dn);
            uint2 *sorted = sc.get<uint2>(dn);
            if (!bd || !bbase || !np || !pbase || !pbin || !bins.ent || !bins.dsc || !bins.tile || !place || !sorted)
                return dcf_set_error(ctx, DCF_ENOMEM, "bins");
            BS_TRY(fill(ctx, bd, 0u, 2 * (int64_t)NB + 1));
            /* distinct slots of a tile where many runs share them: no more slots than pixels, all dense (4096^2 u8 disks 2.12 ms,
             * by runs 2.21, 256^3 1.18 and 1.23; u16 value noise, of longer runs, 1.91 and 1.60) */
            if (sparse) BS_ASSIGN(true, BS_RUNS, 0)
            else if (S <= (unsigned long long)n) BS_ASSIGN(false, BS_SLOTS, 0)
            else BS_ASSIGN(false, BS_RUNS, 0)
            if (is3d) DCF_LAUNCH(ctx, "k_bs_desc", k_bs_desc_count<true>, dim3(nblk(tiles, BS_DTILES)), bl, 0, g, bins, place, bd, be, (int)tiles);
            else DCF_LAUNCH(ctx, "k_bs_desc", k_bs_desc_count<false>, dim3(nblk(tiles, BS_DTILES)), bl, 0, g, bins, place, bd, be, (int)tiles);
            BS_CUB(hipcub::DeviceScan::ExclusiveSum(tmp_, sz_, bd, bbase, (int)(NB + 1), ctx->stream));
            if (is3d) DCF_LAUNCH(ctx, "k_bs_desc", k_bs_desc_place<true>, tg, dim3(64), 0, g, bins, (const uint32_t *)place, (const uint32_t *)bbase, sorted);
            else DCF_LAUNCH(ctx, "k_bs_desc", k_bs_desc_place<false>, tg, dim3(64), 0, g, bins, (const uint32_t *)place, (const uint32_t *)bbase, sorted);
            DCF_LAUNCH(ctx, "k_bs_desc", k_bs_bin_parts, dim3(nblk((int64_t)NB + 1, 256)), bl, 0, (const uint32_t *)bd, (const uint32_t *)be, np, NB);
            BS_CUB(hipcub::DeviceScan::ExclusiveSum(tmp_, sz_, np, pbase, (int)(NB + 1), ctx->stream));
            DCF_LAUNCH(ctx, "k_bs_desc", k_bs_bin_map, dim3(NB), bl, 0, (const uint32_t *)pbase, pbin, first, cnt, (int64_t)S);
            DCF_LAUNCH(ctx, "k_bs_bin", k_bs_bin, dim3(parts), bl, 0, (const uint2 *)bins.ent, (const uint2 *)sorted, (const uint32_t *)bbase,
                       (const uint32_t *)pbase, (const uint32_t *)pbin, NB, first, cnt, (int64_t)S);
            if (is3d) DCF_LAUNCH(ctx, "k_bs_rest", k_bs_rest<true>, tg, dim3(64), 0, g, bins, first, cnt);
            else DCF_LAUNCH(ctx, "k_bs_rest", k_bs_rest<false>, tg, dim3(64), 0, g, bins, first, cnt);
        }
        BsChain ch = sparse ? ch_sparse : ch_nodes;
        if (table.piece > BS_PIECE) {
            /* (wide pieces with few more than BS_SORT pixels each may be more than eight slots per pixel) */
            const int64_t words = (int64_t)(S >> BS_BIN) + 2;
            ch.state = sc.get<unsigned long long>((size_t)words);
            if (!ch.state) return dcf_set_error(ctx, DCF_ENOMEM, "node prefixes");
            BS_TRY(fill(ctx, ch.state, 0u, 2 * words));
        }
        BS_TRY(nodes_of(S, ch));
        DCF_HIP(ctx, hipMemcpyAsync(host + 3, count + 3, 8, hipMemcpyDeviceToHost, ctx->stream));
        DCF_HIP(ctx, hipStreamSynchronize(ctx->stream));
    }

    /* ---- nodes ---- */
    const int64_t K = (int64_t)host[3];
    DevAttr A;
    A.area = own;
    const bool flat = !is3d && t->off[2] == 0;
    BS_TRY(records(ctx, sc, A, grp, flat, K));
    BsLink *link = sc.get<BsLink>((size_t)G);
    BsTotals B;
    B.done = done;
    B.T.area = sc.get<uint32_t>((size_t)G + 1);
    if (!link || !B.T.area) return dcf_set_error(ctx, DCF_ENOMEM, "nodes");
    DCF_LAUNCH(ctx, "k_bs_link", k_bs_link, dim3(nblk((int64_t)G, 256)), bl, 0, (const uint4 *)b.rec, (const uint32_t *)base, (const uint32_t *)nid,
               table, cpar, link, nch, head, B.T.area, (uint32_t)G);

    /* ---- attributes ---- */
#define BS_OWNS(GV)                                                                                                       \
    if (is3d)                                                                                                            \
        DCF_LAUNCH(ctx, "k_bs_own", (k_bs_own<GV, true>), tg, dim3(BS_OWN(GV)), 0, iv, g, t->off[0], t->off[1], t->off[2], (const uint32_t *)slot, \
                   (const uint32_t *)nid, A);                                                                            \
    else                                                                                                                 \
        DCF_LAUNCH(ctx, "k_bs_own", (k_bs_own<GV, false>), tg, dim3(BS_OWN(GV)), 0, iv, g, t->off[0], t->off[1], t->off[2], (const uint32_t *)slot, \
                   (const uint32_t *)nid, A)
    switch (grp) {
    case 0: break;
    case 1: BS_OWNS(1); break;
    case 2: BS_OWNS(2); break;
    case 3: BS_OWNS(3); break;
    default: BS_OWNS(4); break;
    }
    BsPrefix P = {};
    uint32_t *cbase = nullptr;
    int64_t *Es[DCF_MAX_SUMS] = {};
    uint64_t *Emn[3] = {}, *Emx[3] = {};
    bool ok = grp == 0 || (cbase = sc.get<uint32_t>((size_t)K)) != nullptr;
    for (int i = 0; i < A.nsum; i++) ok = ok && (zero_sum(grp, flat, i) || (Es[i] = sc.get<int64_t>((size_t)K + 1)));
    for (int i = 0; A.has_ext && i < 3; i++)
        ok = ok && (Emn[i] = sc.get<uint64_t>((size_t)K)) && (Emx[i] = sc.get<uint64_t>((size_t)K));
    if (!ok) return dcf_set_error(ctx, DCF_ENOMEM, "attribute prefixes");
    P.area = before;
    for (int i = 0; i < DCF_MAX_SUMS; i++) P.s[i] = Es[i];
    for (int i = 0; i < 3; i++) {
        P.mn[i] = Emn[i];
        P.mx[i] = Emx[i];
    }
    if (grp) {
        /* the first node of every node's branch */
        BS_CUB(hipcub::DeviceScan::InclusiveScan(tmp_, sz_, head, cbase, hipcub::Max(), (int)K, ctx->stream));
        BS_TRY(records(ctx, sc, B.T, grp, flat, (int64_t)G));
        BS_TRY(prefixes(ctx, sc, A, cbase, Es, Emn, Emx, K));
    }
#define BS_TOTALS(GV)                                                                                                    \
    DCF_LAUNCH(ctx, "k_bs_totals", k_bs_totals<GV>, dim3(nblk((int64_t)G, 256)), bl, 0, (const BsLink *)link, (const uint32_t *)nch, P, B, (uint32_t)G); \
    DCF_LAUNCH(ctx, "k_bs_join", k_bs_join<GV>, dim3(nblk((int64_t)G, BS_JOIN)), bl, 0, (const BsLink *)link, P, B, A, (uint32_t)G)
    switch (grp) {
    case 0: BS_TOTALS(0); break;
    case 1: BS_TOTALS(1); break;
    case 2: BS_TOTALS(2); break;
    case 3: BS_TOTALS(3); break;
    default: BS_TOTALS(4); break;
    }
    if (grp) BS_TRY(prefixes(ctx, sc, A, cbase, Es, Emn, Emx, K));

    /* ---- results ---- */
    t->grp = -1; /* until the records are whole: an allocation below may fail */
    dcf_free_attr(ctx, t->attr);
    /* For a tree that is there the records are its nodes'.  They are K as here, unless the caller's image (DCF_DEVICE_PTR) no
     * longer holds the pixels of the build: then the records are of no use, but every index below stays in its array */
    const int64_t KT = nodes ? K : t->K;
    BS_TRY(dcf_alloc_attr(ctx, t->attr, grp, KT));
    uint2 *crec = sc.get<uint2>((size_t)K);
    uint32_t *cidx = !nodes || grp ? sc.get<uint32_t>((size_t)KT) : nullptr;
    if (!crec || ((!nodes || grp) && !cidx)) return dcf_set_error(ctx, DCF_ENOMEM, "node records");
    if (!nodes) BS_TRY(fill(ctx, cidx, 0u, KT));
    if (big)
        DCF_LAUNCH(ctx, "k_bs_area", k_bs_area<BS_BIG>, dim3(nblk(K, BS_BIG * 4)), dim3(BS_BIG), 0, (const uint32_t *)own, (const uint32_t *)head,
                   (const uint32_t *)npix, (const int32_t *)cpar, ch_area, crec, nodes ? nullptr : (const uint32_t *)t->p2n,
                   nodes ? nullptr : cidx, K);
    else
        DCF_LAUNCH(ctx, "k_bs_area", k_bs_area<256>, dim3(nblk(K, 1024)), bl, 0, (const uint32_t *)own, (const uint32_t *)head,
                   (const uint32_t *)npix, (const int32_t *)cpar, ch_area, crec, nodes ? nullptr : (const uint32_t *)t->p2n,
                   nodes ? nullptr : cidx, K);
    if (nodes) {
        uint4 *rk = sc.get<uint4>((size_t)(n + 63) / 64);
        int32_t *npar = (int32_t *)dcf_alloc(ctx, (size_t)K * 4);
        float *ngrey = (float *)dcf_alloc(ctx, (size_t)K * 4);
        dcf_release(ctx, t->npar);
        dcf_release(ctx, t->ngrey);
        t->npar = npar;
        t->ngrey = ngrey;
        dcf_release(ctx, t->nroot);
        t->nroot = t->bimg ? (uint32_t *)dcf_alloc(ctx, (size_t)K * 4) : nullptr;
        if (!rk || !npar || !ngrey || (t->bimg && !t->nroot)) return dcf_set_error(ctx, DCF_ENOMEM, "node arrays");
        if (big)
            DCF_LAUNCH(ctx, "k_bs_parent", k_bs_parent<BS_BIG>, dim3(nblk(n, BS_BIG * 16)), dim3(BS_BIG), 0, (const uint32_t *)slot,
                       (const uint32_t *)first, t->parent, rk, ch_roots, n);
        else
            DCF_LAUNCH(ctx, "k_bs_parent", k_bs_parent<256>, dim3(nblk(n, 4096)), bl, 0, (const uint32_t *)slot, (const uint32_t *)first,
                       t->parent, rk, ch_roots, n);
        DCF_LAUNCH(ctx, "k_bs_result", k_bs_result, dim3(nblk(n, 1024)), bl, 0, px, (const uint32_t *)slot, (const uint32_t *)nid, (const uint2 *)crec,
                   (const uint4 *)rk, t->parent, t->p2n, npar, ngrey, t->attr.area, t->nroot, cidx, n);
        t->K = K;
        /* depth bound for the doubling loops: the number of distinct keys */
        t->max_rounds = t->dtype == DCF_U8 ? 9 : (t->dtype == DCF_U16 ? 17 : 33);
    }
#define BS_RECORDS(GV)                                                                                                              \
    DCF_LAUNCH(ctx, "k_bs_records", k_bs_records<GV>, dim3(nblk(KT, 256)), bl, 0, (const uint32_t *)cidx, (const uint32_t *)cbase,  \
               nodes ? nullptr : (const uint2 *)crec, P, t->attr, KT)
    switch (grp) {
    case 0:
        if (!nodes) BS_RECORDS(0);
        break;
    case 1: BS_RECORDS(1); break;
    case 2: BS_RECORDS(2); break;
    case 3: BS_RECORDS(3); break;
    default: BS_RECORDS(4); break;
    }
    t->grp = grp;
    return DCF_OK;
}

/* The tree of t's image: with nodes set, the parent array, pixel -> node map and node arrays; in any case the attribute
 * records of group grp. */
int dcf_basin_build(dcf_tree *t, int grp, bool nodes)
{
    /* saddle edges: in 2D fewer than pixels (peaks and pits take the others) */
    uint64_t edges = 0;
    BS_TRY(basin_build(t, grp, nodes, (uint64_t)t->n + 1024, &edges));
    return edges ? basin_build(t, grp, nodes, edges, &edges) : DCF_OK;
}
