// Host-side check of the blocked sweep as the kernel and the library run it:
// the emulation of block_check.hip (every gathered value the tag that the
// single-step pull reads, every output written once, nothing out of bounds,
// nothing both read and written by one launch) with the kernel's own mapping of
// threads to nodes (block_thread_slab, block_thread_node: z slabs shifted so that
// a wave's nodes start on a line) and with populations padded to whole lines in
// buffers of exactly that size.  Also: a wave lies in one slab, its nodes start on
// a cache line of the lattice and of the ring, and the padding keeps its
// value.  Launches nothing on a GPU.
#define main block_check_main
#include "block_check.hip"
#undef main

static bool fail_at(uint32_t lx, uint32_t ly, uint32_t lz, const char *what)
{
    fprintf(stderr, "%ux%ux%u: %s\n", lx, ly, lz, what);
    return false;
}

static bool check_threads(uint32_t lx, uint32_t ly, uint32_t lz, uint32_t K, int axis, uint32_t W, size_t elem,
                          uint32_t &shifted)
{
    Ctx c;
    c.g = geom(lx, ly, lz);
    const Geom &g = c.g;
    const uint64_t S = padded_stride(g.N, elem), PAD = ~0ull;
    Buf in, out, ring, head;
    in.v.assign(19 * S, PAD);
    out.v.assign(19 * S, PAD);
    ring.v.assign(block_ring_elems(g, axis, K, W, elem), 0);
    head.v.assign(block_head_elems(g, axis, W, elem), 0);
    c.bufs[0] = &in;
    c.bufs[1] = &out;
    c.bufs[2] = &ring;
    c.bufs[3] = &head;
    for (uint64_t n = 0; n < g.N; n++)
        for (int i = 0; i < 19; i++)
            in.v[(uint64_t)i * S + n] = c.tag(0, n, i);
    const StepForce f = {};
    const auto launches =
        block_schedule(g, axis, f, f, K, W, in.v.data(), out.v.data(), ring.v.data(), head.v.data(), S, elem);
    uint64_t out_writes = 0;
    for (const BlockArgs &a : launches) {
        c.reads.clear();
        c.writes.clear();
        c.pending.clear();
        const int s = (a.src.ring == (void *)in.v.data()) ? 0 : 1;
        if (a.slabt % WAVE_LANES != 0 || a.slabt < a.slab)
            return fail_at(lx, ly, lz, "threads of a slab are not whole waves");
        // whole blocks of the launch (256 or 512 threads; the larger covers both)
        const uint64_t nthreads = ((uint64_t)a.slabt * a.count + 511u) / 512u * 512u;
        if (nthreads > 0xffffffffull)
            return fail_at(lx, ly, lz, "thread index beyond 32 bits");
        for (uint32_t t = 0; t < nthreads; t++) {
            const uint32_t sl = block_thread_slab(a, t / WAVE_LANES * WAVE_LANES); // of the wave's first lane
            if (sl != block_thread_slab(a, t))
                return fail_at(lx, ly, lz, "a wave spans two slabs");
            if (sl >= a.count)
                continue;
            const uint32_t sb = block_plane(a, sl);
            const uint32_t w = block_thread_node(a, t, sl, sb);
            if (w >= a.slab)
                continue;
            const BlockRow br = block_row(a, w);
            PlaneRef pl[3];
            block_planes(a, sb, pl);
            const BlockLane l = block_lane(br.ix, br.rs, a.src_nr, (uint32_t)a.src.row_stride, g.lx);
            if (axis == 2)
                gather_all<2>(c, pl, l, br.ix, br.rg, sb, s, std::make_integer_sequence<int, 19>{});
            else
                gather_all<1>(c, pl, l, br.ix, br.rg, sb, s, std::make_integer_sequence<int, 19>{});
            const uint64_t n = node(g, axis, br.ix, br.rg, sb);
            const PlaneRef d = plane_write(a.dst, sb);
            if (axis == 2 && W == 0) { // contiguous slabs: lane k of a wave stores element k of a line
                const uint64_t e = d.off + (uint64_t)(br.rl + a.dst_r0) * d.row_stride + br.ix;
                if ((e - t) % (128 / elem) != 0 || d.stride % (128 / elem) != 0)
                    return fail_at(lx, ly, lz, "a wave's nodes do not start on a line");
                shifted += a.res != 0;
            }
            store(c, d, br.ix, br.rl + a.dst_r0, n, s + 1);
            if (a.dst.ring == (void *)out.v.data())
                out_writes += 19;
            const PlaneRef hd = plane_write_head(a.dst, sb);
            if (hd.buf != nullptr)
                store(c, hd, br.ix, br.rl + a.dst_r0, n, s + 1);
            if (!c.ok)
                return false;
        }
        for (const auto &w : c.writes)
            if (c.reads.count(w))
                return fail_at(lx, ly, lz, "a launch reads and writes the same location");
        if (c.writes.size() != c.pending.size())
            return fail_at(lx, ly, lz, "a launch writes a location twice");
        for (const auto &w : c.pending)
            *w.first = w.second;
    }
    if (out_writes != 19 * g.N)
        return fail_at(lx, ly, lz, "output stores are not one for each value");
    for (int i = 0; i < 19; i++)
        for (uint64_t n = 0; n < S; n++)
            if (out.v[(uint64_t)i * S + n] != (n < g.N ? c.tag(2, n, i) : PAD))
                return fail_at(lx, ly, lz, "output is not step t+2, or the padding was written");
    return true;
}

int main()
{
    // {lx, ly, lz, K, W}: slabs below, at and above a wave, residues 0, 1, 32, 62, 63,
    // windows of every kind
    const uint32_t cases[][5] = {{4, 3, 1, 2, 0},  {4, 3, 2, 2, 0},   {5, 4, 3, 2, 0},   {8, 8, 9, 4, 0},  {13, 5, 9, 4, 0},
                                 {9, 7, 12, 5, 0}, {16, 6, 10, 3, 0}, {31, 4, 8, 4, 0},  {21, 9, 7, 2, 0}, {3, 21, 17, 16, 0},
                                 {7, 5, 33, 8, 0}, {2, 1, 5, 2, 0},   {4, 37, 11, 6, 0}, {2, 5, 75, 32, 0}, {6, 8, 9, 4, 0}, {12, 8, 7, 3, 0}, {10, 16, 5, 2, 0},
                                 {4, 7, 9, 3, 2},  {5, 8, 6, 2, 3},   {3, 10, 4, 4, 1},  {13, 5, 7, 2, 4}, {3, 11, 3, 32, 5}};
    uint32_t shifted = 0;
    for (auto &k : cases)
        for (int axis : {2, 1})
            for (size_t elem : {8, 4, 2})
                if (k[4] < (axis == 2 ? k[1] : k[2]) && !check_threads(k[0], k[1], k[2], k[3], axis, k[4], elem, shifted)) {
                    fprintf(stderr, "K=%u axis %d W=%u elem %zu\n", k[3], axis, k[4], elem);
                    return 1;
                }
    if (shifted == 0) {
        fprintf(stderr, "no slab was shifted\n");
        return 1;
    }
    printf("ok sweep threads\n");
    return 0;
}
