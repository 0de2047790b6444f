// Particle kernels (see particles.h for the methods and their sources).
// Built with -ffp-contract=off: every FP64 operation rounds as written, so
// the CPU oracle's identical expressions give identical bits.
#include <utility>

#include "particles.h"

namespace d3q19 {

namespace {

constexpr int PBLOCK = 256;
// Threads of the kernels that walk a particle's box, one block per particle,
// and the nodes a thread takes per pass: a box of 13^3-15^3 nodes (R = 5)
// takes six or seven passes with 256 threads, each a scan of the block.  The
// main loop runs them beside the collision of large lattices, whose blocks of
// 256 threads leave room for 256 when one of them ends; 512 threads waited for
// the collision's end (250 spheres on 96x384x192: link search 207 us, 114 with
// 256).  With nothing beside them, BOXALONE threads: link search of 20 spheres
// 20.7 us with 256, 11.1 with 1 024, commit and uncovering 9.9 / 6.0 us.
constexpr int BOXBLOCK = 256, BOXALONE = 1024, BOXNODES = 2;
constexpr int IBB_BLOCKS = 4; // blocks per particle for the cut links (~1000-2000 each at R = 5)

// Waves of the kernels that run beside the collision issue ahead of its waves:
// they are few, and the next step waits for them.
__device__ __forceinline__ void ahead_of_collision() { __builtin_amdgcn_s_setprio(3); }

// A periodic index one period at most past the end, or one before the start
// (boxes start in [0, L] and span at most L; neighbours are one node away).
__host__ __device__ inline int wrap(int i, int L) { return i >= L ? i - L : (i < 0 ? i + L : i); }

// Minimum-image offset of a node coordinate from a centre along a periodic axis.
__host__ __device__ inline double min_image(double d, double L)
{
    if (d > 0.5 * L)
        d = d - L;
    else if (d < -0.5 * L)
        d = d + L;
    return d;
}

__host__ __device__ inline void node_offset(const PartGeom &pg, int ix, int iy, int iz, const double *X, double &dx,
                                            double &dy, double &dz)
{
    dx = ((double)ix + 0.5) - X[0];
    dy = min_image(((double)iy + 0.5) - X[1], (double)pg.g.ly);
    dz = min_image(((double)iz + 0.5) - X[2], (double)pg.g.lz);
}

__host__ __device__ inline bool inside(const PartGeom &pg, int ix, int iy, int iz, const double *X)
{
    double dx, dy, dz;
    node_offset(pg, ix, iy, iz, X, dx, dy, dz);
    const double d2 = dx * dx + dy * dy + dz * dz;
    return d2 < pg.R2;
}

__device__ inline uint32_t node_of(const Geom &g, int ix, int iy, int iz)
{
    return (uint32_t)ix + g.lx * ((uint32_t)iy + g.ly * (uint32_t)iz);
}

// Node e of a box in canonical order (x fastest, then y, z).  The quotients
// come from products with reciprocals, exact since (e + 1/2) / d keeps 1/(2d)
// away from every integer: integer divisions took most of a node's
// instructions.
struct BoxNodes {
    Box b;
    int bx, by, bz, bxy, total;
    double ibx, ibxy;
    __device__ inline explicit BoxNodes(const Box &box) : b(box)
    {
        bx = b.x1 - b.x0 + 1;
        by = b.y1 - b.y0 + 1;
        bz = b.z1 - b.z0 + 1;
        bxy = bx * by;
        total = bxy * bz;
        ibx = 1.0 / (double)bx;
        ibxy = 1.0 / (double)bxy;
    }
    __device__ inline uint32_t at(int e, const Geom &g, int &ix, int &iy, int &iz) const
    {
        const int kz = (int)(((double)e + 0.5) * ibxy), r = e - kz * bxy;
        const int ky = (int)(((double)r + 0.5) * ibx);
        ix = b.x0 + (r - ky * bx);
        iy = wrap(b.y0 + ky, (int)g.ly);
        iz = wrap(b.z0 + kz, (int)g.lz);
        return node_of(g, ix, iy, iz);
    }
};

// Block-wide exclusive scan of one int per thread (NT threads, thread
// order), and the block total: an inclusive scan within each wave by lane
// shifts, then the wave totals through LDS.  Integer sums, so the result is
// exact and independent of the scheme.
template <int NT>
__device__ inline int block_scan(int v, int &total)
{
    constexpr int NW = NT / 64;
    __shared__ int wsum[NW];
    const int lane = (int)(threadIdx.x & 63u), wid = (int)(threadIdx.x >> 6);
    int x = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int t = __shfl_up(x, (unsigned)o, 64);
        if (lane >= o)
            x += t;
    }
    if (lane == 63)
        wsum[wid] = x;
    __syncthreads();
    int off = 0, tot = 0;
#pragma unroll
    for (int w = 0; w < NW; w++) {
        const int sw = wsum[w];
        off += w < wid ? sw : 0;
        tot += sw;
    }
    __syncthreads(); // wsum is rewritten by the next call
    total = tot;
    return off + x - v;
}

// Block-wide exclusive scan of BOXNODES counts per thread: the counts of every
// thread's first node come before those of the second.  Two counts of at most
// 18 share an int.
static_assert(BOXNODES == 2 && BOXALONE * 18 < 32768, "two 16-bit sums in an int");
template <int NT>
__device__ inline void box_scan(const int (&v)[BOXNODES], int (&off)[BOXNODES], int &total)
{
    int t;
    const int o = block_scan<NT>(v[0] | v[1] << 16, t);
    const int t0 = t & 0xffff;
    off[0] = o & 0xffff;
    off[1] = t0 + (o >> 16);
    total = t0 + (t >> 16);
}

// The node flags around particle p in LDS, a byte each: what one pass over the
// box reads node by node takes a round trip to memory per pass, and the main
// loop's passes run beside the collision, where one takes 10 us and more (250
// spheres on 96x384x192, link search: 114 us without, 79 with).
enum : uint8_t { FLAG_FLUID = 0, FLAG_MINE = 1, FLAG_OTHER = 2 };
__device__ inline uint8_t flag_of(int solid, int p) { return solid < 0 ? FLAG_FLUID : solid == p ? FLAG_MINE : FLAG_OTHER; }
constexpr int STAGE_FLAGS = 16384; // boxes with more nodes (R above about 10) read memory

// Phase 1: nodes of particle p's previous box still marked p but no longer
// inside become -2-p and join p's refill list (canonical box order).
template <int NT>
__device__ inline void uncover_of(const PartGeom &pg, const PartState &ps, int p, const double *Xold, const double *X)
{
    const BoxNodes box(sphere_box(pg, Xold, 0));
    __shared__ uint8_t mine[STAGE_FLAGS];
    const bool staged = box.total <= STAGE_FLAGS;
    if (staged) {
#pragma unroll 4
        for (int e = threadIdx.x; e < box.total; e += NT) {
            int ix, iy, iz;
            mine[e] = ps.solid[box.at(e, pg.g, ix, iy, iz)] == p;
        }
    } // each thread reads back what it wrote
    int base = 0;
    for (int c0 = 0; c0 < box.total; c0 += NT * BOXNODES) {
        int flag[BOXNODES] = {0, 0}, off[BOXNODES], tot;
        uint32_t n[BOXNODES];
        bool in[BOXNODES];
#pragma unroll
        for (int h = 0; h < BOXNODES; h++) {
            const int e = c0 + h * NT + threadIdx.x;
            int ix, iy, iz;
            n[h] = box.at(e < box.total ? e : 0, pg.g, ix, iy, iz);
            in[h] = e >= box.total || inside(pg, ix, iy, iz, X);
        }
#pragma unroll
        for (int h = 0; h < BOXNODES; h++)
            flag[h] = !in[h] && (staged ? mine[c0 + h * NT + threadIdx.x] != 0 : ps.solid[n[h]] == p);
        box_scan<NT>(flag, off, tot);
#pragma unroll
        for (int h = 0; h < BOXNODES; h++)
            if (flag[h]) {
                ps.solid[n[h]] = -2 - p;
                if (base + off[h] < pg.maxfill)
                    ps.fill_node[(size_t)p * pg.maxfill + base + off[h]] = (int)n[h];
                else
                    atomicOr(ps.overflow, 1);
            }
        base += tot;
    }
    if (threadIdx.x == 0)
        ps.fill_count[p] = base < pg.maxfill ? base : pg.maxfill;
}

__global__ void __launch_bounds__(BOXALONE) k_p_uncover(PartGeom pg, PartState ps, const double *Xold)
{
    uncover_of<BOXALONE>(pg, ps, blockIdx.x, Xold + 3 * blockIdx.x, ps.X + 3 * blockIdx.x);
}

// Commits particle p's move (swaps new positions in, the previous ones are
// kept in Xold, and the new velocities); X and Xo receive the positions.
__device__ inline void commit_of(const PartGeom &pg, const PartState &ps, double *Xold, int p, double (&X)[3],
                                 double (&Xo)[3])
{
    for (int j = 0; j < 3; j++) {
        X[j] = Xold[3 * p + j];
        Xo[j] = ps.X[3 * p + j];
    }
    __syncthreads(); // every thread has read them
    if (threadIdx.x != 0)
        return;
    for (int j = 0; j < 3; j++) {
        Xold[3 * p + j] = Xo[j];
        ps.X[3 * p + j] = X[j];
        ps.V[3 * p + j] = ps.VWnew[3 * p + j];
        ps.W[3 * p + j] = ps.VWnew[3 * pg.np + 3 * p + j];
    }
    if (p == 0)
        *ps.nsteps_done = *ps.nsteps_done + 1;
}

// The main loop's commit and phase 1.
template <int NT>
__global__ void __launch_bounds__(NT) k_p_commit_uncover(PartGeom pg, PartState ps, double *Xold)
{
    ahead_of_collision();
    double X[3], Xo[3];
    commit_of(pg, ps, Xold, blockIdx.x, X, Xo);
    uncover_of<NT>(pg, ps, blockIdx.x, Xo, X);
}

// Phase 2: claim the nodes inside particle p (smallest id wins an overlap).
__global__ void __launch_bounds__(BOXBLOCK) k_p_mark(PartGeom pg, PartState ps)
{
    ahead_of_collision();
    const int p = blockIdx.x;
    const double *X = ps.X + 3 * p;
    const BoxNodes box(sphere_box(pg, X, 0));
    for (int e = threadIdx.x; e < box.total; e += BOXBLOCK) {
        int ix, iy, iz;
        const uint32_t n = box.at(e, pg.g, ix, iy, iz);
        if (inside(pg, ix, iy, iz, X)) {
            // negative (fluid) values compare above every id as unsigned
            atomicMin((unsigned int *)&ps.solid[n], (unsigned int)p);
        }
    }
}

// Phase 3: cut links of particle p: fluid node x, direction i with x + c_i
// inside p.  Canonical order: box node (z, y, x), then direction 1..18.
// A link is at most sqrt(2) long: nodes farther than R + 1.5 from the centre
// cannot reach the sphere.
template <int NT>
__global__ void __launch_bounds__(NT) k_p_links(PartGeom pg, PartState ps)
{
    ahead_of_collision();
    const int p = blockIdx.x;
    const double *X = ps.X + 3 * p;
    const BoxNodes box(sphere_box(pg, X, 1));
    // flags of the box and one node around it: node (ix, iy, iz) of the box at
    // (kx + 1) + sx (ky + 1 + sy (kz + 1)), k from the box's first node
    __shared__ uint8_t flags[STAGE_FLAGS];
    const int sx = box.bx + 2, sy = box.by + 2, sall = sx * sy * (box.bz + 2);
    const bool staged = box.total > 0 && sall <= STAGE_FLAGS;
    if (staged) {
        const double isx = 1.0 / (double)sx, isxy = 1.0 / (double)(sx * sy);
#pragma unroll 4
        for (int e = threadIdx.x; e < sall; e += NT) {
            const int kz = (int)(((double)e + 0.5) * isxy), r = e - kz * (sx * sy);
            const int ky = (int)(((double)r + 0.5) * isx);
            const int jx = box.b.x0 + (r - ky * sx) - 1;
            const bool in = jx >= 0 && jx < (int)pg.g.lx;
            const uint32_t n = node_of(pg.g, in ? jx : box.b.x0, wrap(wrap(box.b.y0 + ky - 1, pg.g.ly), pg.g.ly),
                                       wrap(wrap(box.b.z0 + kz - 1, pg.g.lz), pg.g.lz));
            const uint8_t f = flag_of(ps.solid[n], p);
            flags[e] = in ? f : FLAG_OTHER;
        }
    }
    __syncthreads();
    int base = 0;
    for (int c0 = 0; c0 < box.total; c0 += NT * BOXNODES) {
        uint32_t mask[BOXNODES], n[BOXNODES];
#pragma unroll
        for (int h = 0; h < BOXNODES; h++) {
            const int e = c0 + h * NT + threadIdx.x;
            int ix = 0, iy = 0, iz = 0;
            mask[h] = 0;
            n[h] = 0;
            if (e >= box.total)
                continue;
            n[h] = box.at(e, pg.g, ix, iy, iz);
            double ox, oy, oz;
            node_offset(pg, ix, iy, iz, X, ox, oy, oz);
            const double reach = pg.R + 1.5;
            if (!(ox * ox + oy * oy + oz * oz < reach * reach))
                continue;
            if (staged) {
                const int kz = (int)(((double)e + 0.5) * box.ibxy), r = e - kz * box.bxy;
                const int ky = (int)(((double)r + 0.5) * box.ibx), kx = r - ky * box.bx;
                const int at = (kx + 1) + sx * (ky + 1 + sy * (kz + 1));
                if (flags[at] != FLAG_FLUID)
                    continue;
#pragma unroll
                for (int i = 1; i < 19; i++)
                    if (flags[at + CX[i] + sx * (CY[i] + sy * CZ[i])] == FLAG_MINE)
                        mask[h] |= 1u << i;
            } else {
                // the node's flag and its 18 neighbours' load together; a
                // neighbour beyond a wall reads the node itself (in bounds)
                // and is masked out
                const int ym = wrap(iy - 1, pg.g.ly), yp = wrap(iy + 1, pg.g.ly);
                const int zm = wrap(iz - 1, pg.g.lz), zp = wrap(iz + 1, pg.g.lz);
                const int own = ps.solid[n[h]];
                int sv[19];
#pragma unroll
                for (int i = 1; i < 19; i++) {
                    const int jx = ix + CX[i];
                    const bool in = jx >= 0 && jx < (int)pg.g.lx;
                    const int jy = CY[i] == 0 ? iy : (CY[i] > 0 ? yp : ym);
                    const int jz = CZ[i] == 0 ? iz : (CZ[i] > 0 ? zp : zm);
                    sv[i] = ps.solid[node_of(pg.g, in ? jx : ix, jy, jz)];
                }
                if (own < 0) {
#pragma unroll
                    for (int i = 1; i < 19; i++) {
                        const int jx = ix + CX[i];
                        if (jx >= 0 && jx < (int)pg.g.lx && sv[i] == p)
                            mask[h] |= 1u << i;
                    }
                }
            }
        }
        int cnt[BOXNODES], off[BOXNODES], tot;
#pragma unroll
        for (int h = 0; h < BOXNODES; h++)
            cnt[h] = __builtin_popcount(mask[h]);
        box_scan<NT>(cnt, off, tot);
#pragma unroll
        for (int h = 0; h < BOXNODES; h++) {
            int k = base + off[h];
            for (uint32_t m = mask[h]; m != 0; m &= m - 1) { // set bits, lowest direction first
                if (k < pg.maxlink) {
                    const size_t s = (size_t)p * pg.maxlink + k;
                    ps.link_node[s] = (int)n[h];
                    ps.link_dir[s] = (signed char)__builtin_ctz(m);
                } else {
                    atomicOr(ps.overflow, 1);
                }
                k++;
            }
        }
        base += tot;
    }
    if (threadIdx.x == 0)
        ps.link_count[p] = base < pg.maxlink ? base : pg.maxlink;
}

// Phase 4: the cut-link fraction q of a link of direction i, c_i = (cx, cy,
// cz), from a node at (dx, dy, dz) from the centre: the smaller root of |d + t
// c_i|^2 = R^2, clamped to [0, 1] (1/2 if the line misses the sphere).  |c_i|^2
// is 1 or 2, so the division by it is the exact product with 1 or 1/2.
__device__ inline double link_fraction(const PartGeom &pg, int i, double cx, double cy, double cz, double dx, double dy,
                                       double dz)
{
    const double d2 = dx * dx + dy * dy + dz * dz;
    const double cc = d2 - pg.R2;
    const double a = cx * cx + cy * cy + cz * cz;
    const double inv_a = i <= 6 ? 1.0 : 0.5;
    const double bb = cx * dx + cy * dy + cz * dz;
    const double disc = bb * bb - a * cc;
    double q = (disc >= 0.0) ? (-bb - sqrt(disc)) * inv_a : 0.5;
    if (q < 0.0)
        q = 0.0;
    if (q > 1.0)
        q = 1.0;
    return q;
}

// The fractions of every link, one lane per link.
__global__ void __launch_bounds__(PBLOCK) k_p_linkq(PartGeom pg, PartState ps)
{
    const int p = blockIdx.y;
    const int nl = ps.link_count[p];
    const double *X = ps.X + 3 * p;
    for (int k = blockIdx.x * PBLOCK + threadIdx.x; k < nl; k += gridDim.x * PBLOCK) {
        const size_t s = (size_t)p * pg.maxlink + k;
        const uint32_t n = (uint32_t)ps.link_node[s];
        const int i = ps.link_dir[s];
        const uint32_t qn = fdiv(n, pg.g.dlx);
        const int ix = (int)(n - qn * pg.g.lx);
        const int iz = (int)fdiv(qn, pg.g.dly);
        const int iy = (int)(qn - (uint32_t)iz * pg.g.ly);
        double dx, dy, dz;
        node_offset(pg, ix, iy, iz, X, dx, dy, dz);
        ps.link_q[s] = link_fraction(pg, i, (double)CX[i], (double)CY[i], (double)CZ[i], dx, dy, dz);
    }
}

// Storage access with a run-time direction (2-byte storage scales by
// direction class).
template <int P>
__device__ inline double ld_rt(const typename Prec<P>::S *L, uint64_t N, int i, uint32_t n)
{
    const typename Prec<P>::S v = L[(uint64_t)i * N + n];
    if constexpr (half_storage(P))
        return (double)Prec<P>::to_T_rt(v, i);
    else
        return (double)v;
}

template <int P>
__device__ inline void st_rt(typename Prec<P>::S *L, uint64_t N, int i, uint32_t n, double v)
{
    using S = typename Prec<P>::S;
    if constexpr (half_storage(P))
        L[(uint64_t)i * N + n] = Prec<P>::to_S_rt((float)v, i);
    else
        L[(uint64_t)i * N + n] = (S)v;
}

// Interpolated bounce-back on one cut link of particle p (k < link_count[p]),
// written into the solid node's slot that the fluid node pulls next step;
// the link's momentum-exchange contribution.  With `next` the link's fraction
// is formed here (and stored), else it is there.
template <int P>
__device__ inline void ibb_link(const PartGeom &pg, const PartState &ps, typename Prec<P>::S *L, uint64_t N, int p,
                                int k, bool next)
{
    const size_t s = (size_t)p * pg.maxlink + k;
    const uint32_t n = (uint32_t)ps.link_node[s];
    const int i = ps.link_dir[s];
    const int ib = OPP[i];
    const uint32_t qn = fdiv(n, pg.g.dlx);
    const int ix = (int)(n - qn * pg.g.lx);
    const int iz = (int)fdiv(qn, pg.g.dly);
    const int iy = (int)(qn - (uint32_t)iz * pg.g.ly);
    const double cx = (double)CX[i], cy = (double)CY[i], cz = (double)CZ[i];
    const double w = i <= 6 ? 1.0 / 18.0 : 1.0 / 36.0;

    const double *X = ps.X + 3 * p, *V = ps.V + 3 * p, *W = ps.W + 3 * p;
    double dx, dy, dz;
    node_offset(pg, ix, iy, iz, X, dx, dy, dz);
    double q;
    if (next) {
        q = link_fraction(pg, i, cx, cy, cz, dx, dy, dz);
        ps.link_q[s] = q;
    } else {
        q = ps.link_q[s];
    }
    const double rx = dx + q * cx, ry = dy + q * cy, rz = dz + q * cz; // wall point - centre
    const double uwx = V[0] + (W[1] * rz - W[2] * ry);
    const double uwy = V[1] + (W[2] * rx - W[0] * rz);
    const double uwz = V[2] + (W[0] * ry - W[1] * rx);
    const double cu = cx * uwx + cy * uwy + cz * uwz;

    // Every value either branch may need loads at once, so one memory round
    // trip serves the link: f_i at x, f_opp(i) at x, and flag and f_i of the
    // second fluid node x - c_i behind x (x itself when that lies beyond a
    // wall, so the address stays in bounds; the branch below then ignores it).
    // When x - c_i is a solid node, another link of this launch may be storing
    // into its slots; the value read there is then discarded.
    const int bx_ = ix - CX[i];
    const bool behind_in = (bx_ >= 0 && bx_ < (int)pg.g.lx);
    const uint32_t nb =
        behind_in ? node_of(pg.g, bx_, wrap(iy - CY[i], pg.g.ly), wrap(iz - CZ[i], pg.g.lz)) : n;
    const double fi = ld_rt<P>(L, N, i, n);
    const double fib = ld_rt<P>(L, N, ib, n);
    const int solid_b = ps.solid[nb];
    const double fb = ld_rt<P>(L, N, i, nb);
    double g;
    if (q < 0.5) {
        if (behind_in && solid_b < 0)
            g = (2.0 * q) * fi + (1.0 - 2.0 * q) * fb - 6.0 * w * cu;
        else
            g = fi - 6.0 * w * cu;
    } else {
        g = (1.0 / (2.0 * q)) * fi + ((2.0 * q - 1.0) / (2.0 * q)) * fib - (3.0 / q) * w * cu;
    }
    // the solid node x + c_i: its slot ib is what x pulls for direction ib
    const uint32_t ns = node_of(pg.g, ix + CX[i], wrap(iy + CY[i], pg.g.ly), wrap(iz + CZ[i], pg.g.lz));
    st_rt<P>(L, N, ib, ns, g);

    // momentum exchange with full populations f = shifted + w*rho0
    const double ff = fi + w, gf = g + w;
    const double px = ff * (cx - uwx) + gf * (cx + uwx);
    const double py = ff * (cy - uwy) + gf * (cy + uwy);
    const double pz = ff * (cz - uwz) + gf * (cz + uwz);
    double *c = ps.link_contrib + (size_t)p * 6 * pg.maxlink + k;
    const size_t m = pg.maxlink;
    c[0] = px;
    c[m] = py;
    c[2 * m] = pz;
    c[3 * m] = ry * pz - rz * py;
    c[4 * m] = rz * px - rx * pz;
    c[5 * m] = rx * py - ry * px;
}

// Uncovered nodes become ordinary fluid once every refill has read its
// neighbours.
__device__ inline void settle_of(const PartState &ps, const PartGeom &pg, int p, int first, int step)
{
    const int nf = ps.fill_count[p];
    for (int k = first; k < nf; k += step) {
        const uint32_t n = (uint32_t)ps.fill_node[(size_t)p * pg.maxfill + k];
        if (ps.solid[n] == -2 - p)
            ps.solid[n] = -1;
    }
}

__global__ void k_p_settle(PartGeom pg, PartState ps) { settle_of(ps, pg, blockIdx.x, threadIdx.x, blockDim.x); }

// Every cut link: IBB_BLOCKS blocks per particle stride over its links.  With
// `next`, in the main loop after its first step, the fractions are formed here
// and the first block settles the nodes refilled before (the bounce-back reads
// flags by their sign, which settling keeps): two launches less in the chain
// between two steps.
template <int P>
__global__ void __launch_bounds__(PBLOCK) k_p_ibb(PartGeom pg, PartState ps, void *Lv, int next)
{
    using S = typename Prec<P>::S;
    const int p = blockIdx.y;
    if (next && blockIdx.x == 0)
        settle_of(ps, pg, p, threadIdx.x, PBLOCK);
    const int nl = ps.link_count[p];
    S *L = (S *)Lv;
    const uint64_t N = pg.g.S; // population stride
    for (int k = blockIdx.x * PBLOCK + threadIdx.x; k < nl; k += gridDim.x * PBLOCK)
        ibb_link<P>(pg, ps, L, N, p, k, next != 0);
}

// Sums in a fixed order over the 64 lanes of a wave: lane l adds terms l,
// l+64, l+128, ... in increasing order, then the 64 partials are added pairwise
// (l += l + 32, l += l + 16, ..., l += l + 1).  The CPU oracle sums in the
// same order, so results agree bit for bit.  Lane 0 gets the sum.
constexpr int SUMW = 64;

template <int C>
__device__ inline void lane_tree(double (&v)[C])
{
#pragma unroll
    for (int off = SUMW / 2; off > 0; off >>= 1)
#pragma unroll
        for (int j = 0; j < C; j++)
            v[j] = v[j] + __shfl_down(v[j], off);
}

// Force and torque of particle p from the per-link contributions: components
// j0 and j0 + 1 of (force, torque), by one wave.  Eight terms of a lane load
// together: one round trip per term took 56 us for 250 spheres beside the
// collision.
__device__ inline void sum_of(const PartGeom &pg, const PartState &ps, int p, int j0, double (&f)[2])
{
    constexpr int U = 8;
    const int l = threadIdx.x & (SUMW - 1);
    const int nl = ps.link_count[p];
    const double *c = ps.link_contrib + ((size_t)p * 6 + j0) * pg.maxlink;
    f[0] = f[1] = 0.0;
    for (int k0 = l; k0 < nl; k0 += U * SUMW) {
        double v[2][U];
#pragma unroll
        for (int u = 0; u < U; u++)
#pragma unroll
            for (int j = 0; j < 2; j++)
                v[j][u] = k0 + u * SUMW < nl ? c[j * (size_t)pg.maxlink + k0 + u * SUMW] : 0.0;
#pragma unroll
        for (int u = 0; u < U; u++)
            if (k0 + u * SUMW < nl) {
                f[0] = f[0] + v[0][u];
                f[1] = f[1] + v[1][u];
            }
    }
    lane_tree(f);
    if (l == 0)
        for (int j = 0; j < 2; j++)
            (j0 + j < 3 ? ps.FH + 3 * p : ps.TQ + 3 * p - 3)[j0 + j] = f[j];
}

// One block of three waves per particle, two components each.
__global__ void __launch_bounds__(3 * SUMW) k_p_sum(PartGeom pg, PartState ps)
{
    double f[2];
    sum_of(pg, ps, blockIdx.x, 2 * (threadIdx.x / SUMW), f);
}

// Contact force magnitude of Feng & Michaelides (2005) eq. 28 for the gap h
// and range zeta: stf0 ((zeta - h)/zeta)^2 below zeta, plus stf1 (-h/zeta)
// on overlap (h < 0).
__device__ inline double contact_mag(double h, double zeta, double stf0, double stf1)
{
    if (!(h < zeta))
        return 0.0;
    const double r = (zeta - h) / zeta;
    double m = stf0 * (r * r);
    if (h < 0.0)
        m = m + stf1 * ((-h) / zeta);
    return m;
}

// Coefficient of the approach velocity in the lubrication correction of
// Nguyen & Ladd (2002): -6 pi mu a^2 (1/h - 1/hc), the gap no smaller than
// lub_min, zero at or beyond hc or without viscosity (mu = rho0 nu, rho0 = 1).
__device__ inline double lub_coef(double h, double a, const PartGeom &pg)
{
    if (!(pg.visc > 0.0) || !(h < pg.lub_cut))
        return 0.0;
    const double he = h > pg.lub_min ? h : pg.lub_min;
    return -6.0 * 3.14159265358979323846 * pg.visc * (a * a) * (1.0 / he - 1.0 / pg.lub_cut);
}

// Contact and lubrication forces of particle p from the others (f6), by one
// wave whose lanes split them (q = l, l+64, ...).  Lane 0 gets the sums.
__device__ inline void pairs_of(const PartGeom &pg, const PartState &ps, int p, double (&f6)[6])
{
    const int l = threadIdx.x & (SUMW - 1);
    const double Ly = (double)pg.g.ly, Lz = (double)pg.g.lz;
    const double *Xp = ps.X + 3 * p, *Vp = ps.V + 3 * p;
    for (int j = 0; j < 6; j++)
        f6[j] = 0.0;
    for (int q = l; q < pg.np; q += SUMW) {
        if (q == p)
            continue;
        const double *Xq = ps.X + 3 * q, *Vq = ps.V + 3 * q;
        const double ddx = Xp[0] - Xq[0];
        const double ddy = min_image(Xp[1] - Xq[1], Ly);
        const double ddz = min_image(Xp[2] - Xq[2], Lz);
        const double dist = sqrt(ddx * ddx + ddy * ddy + ddz * ddz);
        if (!(dist > 0.0))
            continue;
        const double h = dist - 2.0 * pg.R;
        const double nx = ddx / dist, ny = ddy / dist, nz = ddz / dist;
        const double mag = contact_mag(h, pg.mingap, pg.stf0, pg.stf1);
        const double un = (Vp[0] - Vq[0]) * nx + (Vp[1] - Vq[1]) * ny + (Vp[2] - Vq[2]) * nz;
        const double lub = lub_coef(h, 0.5 * pg.R, pg) * un;
        f6[0] = f6[0] + mag * nx;
        f6[1] = f6[1] + mag * ny;
        f6[2] = f6[2] + mag * nz;
        f6[3] = f6[3] + lub * nx;
        f6[4] = f6[4] + lub * ny;
        f6[5] = f6[5] + lub * nz;
    }
    lane_tree(f6);
}

// Walls and FP64 integration of component j of particle p, whose contact and
// lubrication sums are fc and fl and whose hydrodynamic force and torque are
// FH and TQ.  Every particle reads the positions and velocities before the
// move; the new ones are staged (Xold, VWnew) and swapped in by commit_of.
__device__ inline void move_of(const PartGeom &pg, const PartState &ps, double *Xold, int p, int j, double fc, double fl,
                               double FH, double TQ)
{
    const int k = 3 * p + j;
    const double v0 = ps.V[k], w0 = ps.W[k], x0 = ps.X[k];
    const double FHp = ps.FHprev[k], TQp = ps.TQprev[k], Ap = ps.Aprev[k], ALp = ps.ALprev[k], TH = ps.TH[k];
    const bool first = (*ps.nsteps_done == 0);
    if (j == 0) {
        // walls at x = 0 and x = lx: the mirror image lies twice the distance away
        const double dlo = x0, dhi = (double)pg.g.lx - x0;
        fc = fc + contact_mag(2.0 * dlo - 2.0 * pg.R, pg.mingap_w, pg.stf0_w, pg.stf1_w);
        fc = fc - contact_mag(2.0 * dhi - 2.0 * pg.R, pg.mingap_w, pg.stf0_w, pg.stf1_w);
        fl = fl + lub_coef(dlo - pg.R, pg.R, pg) * v0;
        fl = fl + lub_coef(dhi - pg.R, pg.R, pg) * v0;
    }
    ps.FC[k] = fc;
    ps.FL[k] = fl;
    const double fh = first ? FH : 0.5 * (FH + FHp);
    const double tq = first ? TQ : 0.5 * (TQ + TQp);
    ps.FHprev[k] = FH;
    ps.TQprev[k] = TQ;
    double ftot = fh + fc + fl;
    if (pg.pressure_force)
        ftot = ftot + pg.volume * (j == 0 ? pg.fx : j == 1 ? pg.fy : pg.fz);
    const double a = ftot / pg.mass;
    const double al = tq / pg.inertia;
    const double Vn = first ? v0 + a : v0 + (1.5 * a - 0.5 * Ap);
    const double Wn = first ? w0 + al : w0 + (1.5 * al - 0.5 * ALp);
    double Xn = x0 + 0.5 * (v0 + Vn);
    ps.TH[k] = TH + 0.5 * (w0 + Wn);
    ps.Aprev[k] = a;
    ps.ALprev[k] = al;
    if (j > 0) {
        const double L = (double)(j == 1 ? pg.g.ly : pg.g.lz);
        if (Xn >= L)
            Xn = Xn - L;
        else if (Xn < 0.0)
            Xn = Xn + L;
    }
    // a diverged run: flag it (sphere_box then gives empty boxes for such a
    // particle, so no kernel indexes from it)
    if (!((Xn - Xn == 0.0) && (Vn - Vn == 0.0) && (Wn - Wn == 0.0)))
        atomicOr(ps.overflow, 2);
    Xold[k] = Xn;
    ps.VWnew[k] = Vn;
    ps.VWnew[3 * pg.np + k] = Wn;
}

// One wave per particle; lanes 0-2 integrate a component each.
__global__ void __launch_bounds__(SUMW) k_p_move(PartGeom pg, PartState ps, double *Xold)
{
    const int p = blockIdx.x, l = threadIdx.x;
    double f[6];
    pairs_of(pg, ps, p, f);
#pragma unroll
    for (int j = 0; j < 6; j++)
        f[j] = __shfl(f[j], 0);
    if (l < 3)
        move_of(pg, ps, Xold, p, l, f[l], f[3 + l], ps.FH[3 * p + l], ps.TQ[3 * p + l]);
}

// The main loop's sums and move, four waves per particle: three sum two
// components each while the fourth works on the pairs (one wave for all of it
// took 85 us beside the collision, 35 now).
__global__ void __launch_bounds__(4 * SUMW) k_p_sum_move(PartGeom pg, PartState ps, double *Xold)
{
    ahead_of_collision();
    const int p = blockIdx.x, l = threadIdx.x & (SUMW - 1), w = threadIdx.x / SUMW;
    __shared__ double s[12]; // force, torque, contact, lubrication
    if (w < 3) {
        double f[2];
        sum_of(pg, ps, p, 2 * w, f);
        if (l == 0) {
            s[2 * w] = f[0];
            s[2 * w + 1] = f[1];
        }
    } else {
        double f[6];
        pairs_of(pg, ps, p, f);
        if (l == 0)
            for (int j = 0; j < 6; j++)
                s[6 + j] = f[j];
    }
    __syncthreads();
    if (threadIdx.x < 3)
        move_of(pg, ps, Xold, p, l, s[6 + l], s[9 + l], s[l], s[3 + l]);
}

__global__ void __launch_bounds__(SUMW) k_p_commit(PartGeom pg, PartState ps, double *Xold)
{
    double X[3], Xo[3];
    commit_of(pg, ps, Xold, blockIdx.x, X, Xo);
}

// macrovar's solid branch (Channel-Flow/collision.f90:420-459): nodes inside
// particle p carry the rigid-body velocity V + W x r (r from the centre,
// minimum image in y and z) and rho = rhopart, less the pending avedensity
// offset, which the reference subtracts from every node (:508).  One block
// per particle strides over its box.
__global__ void __launch_bounds__(PBLOCK) k_p_solid_fields(PartGeom pg, PartState ps, double rho_off, double *rho,
                                                            double *ux, double *uy, double *uz)
{
    const int p = blockIdx.x;
    const double *X = ps.X + 3 * p, *V = ps.V + 3 * p, *W = ps.W + 3 * p;
    const BoxNodes box(sphere_box(pg, X, 0));
    for (int t = threadIdx.x; t < box.total; t += PBLOCK) {
        int ix, iy, iz;
        const uint32_t n = box.at(t, pg.g, ix, iy, iz);
        if (ps.solid[n] != p)
            continue;
        double dx, dy, dz;
        node_offset(pg, ix, iy, iz, X, dx, dy, dz);
        ux[n] = V[0] + (W[1] * dz - W[2] * dy);
        uy[n] = V[1] + (W[2] * dx - W[0] * dz);
        uz[n] = V[2] + (W[0] * dy - W[1] * dx);
        rho[n] = pg.rhopart - rho_off;
    }
}

// Refill: nodes uncovered by particle p get the equilibrium of the wall
// velocity there and the mean density of their settled fluid neighbours.
// Refill of the uncovered nodes of particle p, REFILL_NODES nodes per wave
// pass, the passes dealt to the block's waves in turn.  Lane 18 t + (j - 1) of
// a pass serves node t of the pass and its neighbour x + c_j (j = 1..18): it
// loads that neighbour's flag and, for a fluid neighbour inside the walls, its
// 19 populations, and sums them in population order (its density).  Every
// lane of the node then adds the 18 densities in j order from the wave's LDS,
// as one thread walking the neighbours would, so rho, and with it every
// stored value, does not depend on the lane layout.  The node gets the
// equilibrium at rho and the wall velocity V + W x r; lane j stores
// population j, lane 1 also population 0.  A node claimed by another particle
// since it was listed is left alone.
constexpr int REFILL_NODES = 3; // 3 x 18 = 54 of the 64 lanes

// Orders a wave's LDS stores before its later loads by other lanes: the LDS
// serves one wave's instructions in order, so only the compiler is held.
__device__ __forceinline__ void wave_lds_order()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <int P, int NT>
__device__ inline void refill_of(const PartGeom &pg, const PartState &ps, typename Prec<P>::S *L, int p)
{
    const uint64_t N = pg.g.S; // population stride
    const int nf = ps.fill_count[p];
    const int l = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const int t = l / 18, j = l % 18 + 1;
    __shared__ double rs_all[NT / 64][REFILL_NODES][18];
    __shared__ int ok_all[NT / 64][REFILL_NODES][18];
    auto &rs = rs_all[wid];
    auto &ok = ok_all[wid];
    for (int k0 = wid * REFILL_NODES; k0 < nf; k0 += NT / 64 * REFILL_NODES) {
        const int k = k0 + t;
        const bool lane = t < REFILL_NODES && k < nf;
        uint32_t n = 0;
        int ix = 0, iy = 0, iz = 0;
        bool mine = false;
        if (lane) {
            n = (uint32_t)ps.fill_node[(size_t)p * pg.maxfill + k];
            mine = ps.solid[n] == -2 - p;
            const uint32_t qn = fdiv(n, pg.g.dlx);
            ix = (int)(n - qn * pg.g.lx);
            iz = (int)fdiv(qn, pg.g.dly);
            iy = (int)(qn - (uint32_t)iz * pg.g.ly);
        }
        wave_lds_order(); // the previous pass has been read
        if (lane && mine) {
            double r = 0.0;
            int use = 0;
            const int jx = ix + CX[j];
            if (jx >= 0 && jx < (int)pg.g.lx) {
                const uint32_t m = node_of(pg.g, jx, wrap(iy + CY[j], pg.g.ly), wrap(iz + CZ[j], pg.g.lz));
                if (ps.solid[m] == -1) {
                    double f[19];
#pragma unroll
                    for (int i = 0; i < 19; i++)
                        f[i] = ld_rt<P>(L, N, i, m);
                    r = f[0];
#pragma unroll
                    for (int i = 1; i < 19; i++)
                        r = r + f[i];
                    use = 1;
                }
            }
            rs[t][j - 1] = r;
            ok[t][j - 1] = use;
        }
        wave_lds_order();
        if (lane && mine) {
            double rsum = 0.0;
            int cnt = 0;
            for (int jj = 0; jj < 18; jj++)
                if (ok[t][jj]) {
                    rsum = rsum + rs[t][jj];
                    cnt++;
                }
            const double rho = cnt > 0 ? rsum / (double)cnt : 0.0;
            const double *X = ps.X + 3 * p, *V = ps.V + 3 * p, *W = ps.W + 3 * p;
            double dx, dy, dz;
            node_offset(pg, ix, iy, iz, X, dx, dy, dz);
            const double ux = V[0] + (W[1] * dz - W[2] * dy);
            const double uy = V[1] + (W[2] * dx - W[0] * dz);
            const double uz = V[2] + (W[0] * dy - W[1] * dx);
            double usqr = ux * ux + uy * uy + uz * uz;
            usqr = 1.5 * usqr;
            if (j == 1)
                st_rt<P>(L, N, 0, n, (1.0 / 3.0) * (rho - usqr));
            const double G = (double)CX[j] * ux + (double)CY[j] * uy + (double)CZ[j] * uz;
            const double w = j <= 6 ? 1.0 / 18.0 : 1.0 / 36.0;
            st_rt<P>(L, N, j, n, w * (rho + 3.0 * G + 4.5 * G * G - usqr));
        }
    }
}

template <int P>
__global__ void __launch_bounds__(PBLOCK) k_p_refill(PartGeom pg, PartState ps, void *Lv)
{
    refill_of<P, PBLOCK>(pg, ps, (typename Prec<P>::S *)Lv, blockIdx.x);
}

// The collision's flags where the last classification can have changed the
// sign of solid: particle p's box before it and its box now.
template <int P>
__device__ inline void inside_of(const PartGeom &pg, const PartState &ps, int p)
{
    InsideFlag<P> *const inside = (InsideFlag<P> *)ps.inside;
    for (int old = 0; old < 2; old++) {
        const BoxNodes box(sphere_box(pg, ps.X + 3 * ((size_t)old * pg.np + p), 0));
        for (int e = threadIdx.x; e < box.total; e += BOXBLOCK) {
            int ix, iy, iz;
            const uint32_t n = box.at(e, pg.g, ix, iy, iz);
            inside[n] = ps.solid[n] >= 0;
        }
    }
}

template <int P>
__global__ void __launch_bounds__(BOXBLOCK) k_p_inside(PartGeom pg, PartState ps)
{
    inside_of<P>(pg, ps, blockIdx.x);
}

// What the main loop does between two steps besides the bounce-back: the
// refill and the collision's flags, neither of which reads what the other
// writes.
template <int P>
__global__ void __launch_bounds__(BOXBLOCK) k_p_refill_inside(PartGeom pg, PartState ps, void *Lv)
{
    if ((int)blockIdx.x < pg.np)
        refill_of<P, BOXBLOCK>(pg, ps, (typename Prec<P>::S *)Lv, blockIdx.x);
    else
        inside_of<P>(pg, ps, (int)blockIdx.x - pg.np);
}

} // namespace

template <int P>
hipError_t PartLaunch<P>::inside(const PartGeom &pg, const PartState &ps, hipStream_t s)
{
    hipLaunchKernelGGL((k_p_inside<P>), dim3(pg.np), dim3(BOXBLOCK), 0, s, pg, ps);
    return hipGetLastError();
}

hipError_t part_solid_fields(const PartGeom &pg, const PartState &ps, double rho_off, double *rho, double *ux,
                             double *uy, double *uz, hipStream_t s)
{
    hipLaunchKernelGGL(k_p_solid_fields, dim3(pg.np), dim3(PBLOCK), 0, s, pg, ps, rho_off, rho, ux, uy, uz);
    return hipGetLastError();
}

hipError_t part_sum(const PartGeom &pg, const PartState &ps, hipStream_t s)
{
    hipLaunchKernelGGL(k_p_sum, dim3(pg.np), dim3(3 * SUMW), 0, s, pg, ps);
    return hipGetLastError();
}

hipError_t part_move(const PartGeom &pg, const PartState &ps, hipStream_t s)
{
    double *Xold = ps.X + 3 * (size_t)pg.np;
    hipLaunchKernelGGL(k_p_move, dim3(pg.np), dim3(SUMW), 0, s, pg, ps, Xold);
    hipLaunchKernelGGL(k_p_commit, dim3(pg.np), dim3(SUMW), 0, s, pg, ps, Xold);
    return hipGetLastError();
}

static void launch_settle(const PartGeom &pg, const PartState &ps, hipStream_t s)
{
    hipLaunchKernelGGL(k_p_settle, dim3(pg.np), dim3(64), 0, s, pg, ps);
}

static void launch_mark_links(const PartGeom &pg, const PartState &ps, bool aside, hipStream_t s)
{
    hipLaunchKernelGGL(k_p_mark, dim3(pg.np), dim3(BOXBLOCK), 0, s, pg, ps);
    if (aside)
        hipLaunchKernelGGL(k_p_links<BOXBLOCK>, dim3(pg.np), dim3(BOXBLOCK), 0, s, pg, ps);
    else
        hipLaunchKernelGGL(k_p_links<BOXALONE>, dim3(pg.np), dim3(BOXALONE), 0, s, pg, ps);
}

static void launch_fractions(const PartGeom &pg, const PartState &ps, hipStream_t s)
{
    hipLaunchKernelGGL(k_p_linkq, dim3(IBB_BLOCKS, pg.np), dim3(PBLOCK), 0, s, pg, ps);
}

hipError_t part_classify(const PartGeom &pg, const PartState &ps, int first, hipStream_t s)
{
    // ps.Aprev is not touched; Xold lives after X in the state (see lbm_capi)
    if (!first)
        hipLaunchKernelGGL(k_p_uncover, dim3(pg.np), dim3(BOXALONE), 0, s, pg, ps, ps.X + 3 * (size_t)pg.np);
    launch_mark_links(pg, ps, false, s);
    launch_fractions(pg, ps, s);
    return hipGetLastError();
}

hipError_t part_advance(const PartGeom &pg, const PartState &ps, bool aside, hipStream_t s)
{
    double *Xold = ps.X + 3 * (size_t)pg.np;
    hipLaunchKernelGGL(k_p_sum_move, dim3(pg.np), dim3(4 * SUMW), 0, s, pg, ps, Xold);
    if (aside)
        hipLaunchKernelGGL(k_p_commit_uncover<BOXBLOCK>, dim3(pg.np), dim3(BOXBLOCK), 0, s, pg, ps, Xold);
    else
        hipLaunchKernelGGL(k_p_commit_uncover<BOXALONE>, dim3(pg.np), dim3(BOXALONE), 0, s, pg, ps, Xold);
    launch_mark_links(pg, ps, aside, s);
    return hipGetLastError();
}

hipError_t part_finish(const PartGeom &pg, const PartState &ps, hipStream_t s)
{
    launch_fractions(pg, ps, s);
    launch_settle(pg, ps, s);
    return hipGetLastError();
}

template <int P>
hipError_t PartLaunch<P>::ibb(const PartGeom &pg, const PartState &ps, void *L, bool next, hipStream_t s)
{
    hipLaunchKernelGGL((k_p_ibb<P>), dim3(IBB_BLOCKS, pg.np), dim3(PBLOCK), 0, s, pg, ps, L, (int)next);
    return hipGetLastError();
}

template <int P>
hipError_t PartLaunch<P>::refill(const PartGeom &pg, const PartState &ps, void *L, hipStream_t s)
{
    hipLaunchKernelGGL((k_p_refill<P>), dim3(pg.np), dim3(PBLOCK), 0, s, pg, ps, L);
    launch_settle(pg, ps, s);
    return hipGetLastError();
}

template <int P>
hipError_t PartLaunch<P>::refill_inside(const PartGeom &pg, const PartState &ps, void *L, hipStream_t s)
{
    hipLaunchKernelGGL((k_p_refill_inside<P>), dim3(2 * pg.np), dim3(BOXBLOCK), 0, s, pg, ps, L);
    return hipGetLastError();
}

template struct PartLaunch<0>;
template struct PartLaunch<1>;
template struct PartLaunch<2>;
template struct PartLaunch<3>;

} // namespace d3q19
