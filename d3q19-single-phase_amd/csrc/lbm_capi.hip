// C ABI of liblbm (include/lbm.h): handle, device memory, and the mapping of
// the reference's subroutines onto kernel launches.
//
// Macroscopic fields.  The reference keeps rho, ux, uy, uz as module arrays
// that collision_MRT reads (Channel-Flow/collision.f90:56-59) and macrovar,
// rhoupdat, avedensity, initvel/initpop write.  In the main loop they always
// hold macrovar of the current f, so the step kernel recomputes them from the
// populations it already gathers and the arrays are never touched.  The
// handle tracks what the arrays logically hold:
//   FROM_CUR   macrovar(F_cur) with rho - rho_off  (nothing stored)
//   FROM_PREV  macrovar(F_prev) with rho - rho_off (after a collision that
//              was not followed by macrovar; F_prev is still in the other
//              lattice)
//   ARRAYS     the device arrays hold the values
// and materialises the arrays only when a call needs stored values.
#include <hip/hip_runtime.h>

#include <math.h>
#include <stdarg.h>
#include <stdio.h>
#include <string.h>

#include <algorithm>
#include <cmath>
#include <mutex>
#include <vector>

#include "blocked.h"
#include "hostcopy.h"
#include "kernels.h"
#include "lbm.h"
#include "particles.h"
#include "mlp_train.h"

using namespace d3q19;

namespace {

thread_local char g_err[512] = "";

int fail(int code, const char *fmt, ...)
{
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof(g_err), fmt, ap);
    va_end(ap);
    return code;
}

#define HIP_TRY(call)                                                                                     \
    do {                                                                                                  \
        hipError_t e_ = (call);                                                                           \
        if (e_ != hipSuccess)                                                                             \
            return fail(LBM_ERR_HIP, "%s failed: %s (%s:%d)", #call, hipGetErrorString(e_), __FILE__, __LINE__); \
    } while (0)

enum MacroState { FROM_CUR = 0, FROM_PREV = 1, ARRAYS = 2 };

constexpr uint32_t RED_BLOCKS = 2048;   // partial sums per reduction
constexpr uint32_t DIAG_BLOCKS = 1024;  // partials per quantity of diag
constexpr uint32_t PLANE_CHUNKS = 512;  // row chunks for plane sums
constexpr size_t ERR_BYTES = (ERR_SLOTS * ERR_STRIDE + 1) * sizeof(unsigned long long); // lbm_channel::errbits
constexpr size_t STAGE_BYTES = HOST_WORKERS * HOST_DEPTH * HOST_SLICE; // device side of the copy slices

// Scratch of lbm_mass_sum_noalloc: the per-block partial sums of the mass
// reduction, 16 KiB per GPU, held until the process ends.  Host code never passes `scratch` itself
// to a kernel: it uses the device address that hipGetSymbolAddress returns
// for the current device (scratch_ptr), kept per device.
constexpr uint32_t NOALLOC_PARTIALS = RED_BLOCKS;
constexpr int MAX_DEVICES = 64;
double *g_scratch_ptr[MAX_DEVICES];
std::mutex g_scratch_mu;

} // namespace

static __device__ __align__(256) double scratch[NOALLOC_PARTIALS];

struct lbm_channel {
    lbm_config cfg;
    Geom g;
    int prec;
    size_t elem; // bytes per stored population
    void *lat[2];
    int cur;       // lattice holding P of the current state
    bool have_prev;
    bool fresh;    // no step or field assignment yet
    double *mac[4]; // rho, ux, uy, uz (allocated on first use)
    MacroState ms;
    double rho_off;
    ForceSpec fc;       // the force arrays' contents: FORCING (uniform) or FORCINGP
    ForceSpec fm;       // the force that the fields FROM_CUR / FROM_PREV are formed with
    double *ftab;       // FORCINGP factor tables (allocated on first use)
    hipStream_t stream;
    double *partials;   // 2*RED_BLOCKS doubles, then PLANE_CHUNKS*NPLANE*lx doubles
    double *red_out;    // 2 doubles + NPLANE*lx doubles of final sums
    unsigned long long *errbits; // ERR_SLOTS maxima of rhoupdat, zero between calls; behind them the stop word of lbm_prerelax
    unsigned long long *errout;  // their maxima, pinned (allocated on first use): PRE_ITERS words of lbm_prerelax, one of rhoupdat
    double *small;      // NPLANE*lx doubles (64 at least) for results the host reads (ensure_small)
    bool small_pinned;  // the device can store into it
    double *stat_acc;   // NPLANE*lx running sums
    long long stat_n;
    double *fstat_acc;  // NPLANE*(lx/2) running sums of the box-filtered fields (allocated on first use)
    long long fstat_n;
    char *stage;        // STAGE_BYTES: one device slice for every slot of the host copies
    hipEvent_t ev[2];
    struct Part *part;  // rigid particles (nullptr without)
    hipStream_t pstream; // lbm_run_particles: the force sums and beads_move beside the collision
    hipEvent_t pev[2];   // its fork (after the bounce-back) and join (before the refill)
    int pstreams;        // streams of lbm_run_particles: 1, 2 or by the lattice's size (0)
    float *mlp;         // learned closure parameters on the device (nullptr: plain MRT)
    float mlp_inv_ystar, mlp_yscale;
    int runs;           // step kernel: 1 = vector runs where the shape allows, 0 = one node per thread
    int w32;            // step kernel: 1 = 32-bit pull offsets where N allows (default), 2 = between adjacent rows only
    uint32_t bK;        // two-step blocked sweep: slabs per chunk (0 = single steps only)
    int baxis;          // its sweep axis: 2 = z (slabs lx*ly), 1 = y (slabs lx*lz)
    uint32_t bW;        // rows per window of its slabs (0 = whole slabs)
    bool bskip;         // the lattice is small: pairs run as single steps although bK > 0
    int bforced;        // lbm_run_forcingp also pairs steps whose force varies over the nodes
    void *bring, *bhead; // its slab ring and head buffer (allocated on first use)
    bool ave_pending;   // lbm_run_particles: avedensity due once the next bounce-back has run
    // Per-call pairing: collision_MRT calls whose launch is deferred (0-2) so
    // that collision, macrovar, collision, macrovar runs as one blocked pair;
    // pend_mac: a fields-only macrovar followed the first; defer: enabled
    // (LBM_DEFER=0 at lbm_create turns it off)
    int pend;
    bool pend_mac;
    int defer;
};

struct lbm_trainer {
    int device;
    hipStream_t stream;
    long long capacity, count;
    float *feat, *target;   // capacity x 10, capacity
    float *w, *m, *v;       // LBM_MLP_TOTAL parameters, Adam moments
    float *partial, *grad;  // per-block partial gradients, summed gradient (+ loss)
    float *small;           // MLP_TOTAL floats for results the host reads
    bool small_pinned;      // the device can store into it
    uint32_t max_waves;
    int step;
    int target_mode; // LBM_TARGET_LOCAL or LBM_TARGET_PLANE for lbm_trainer_add_filtered
};

// Particle set on the device (see particles.h).
constexpr size_t PART_STATE = 24; // doubles a particle in the block that ps.X starts
struct Part {
    PartGeom pg;
    PartState ps;
    std::vector<void *> allocs;
    std::vector<double> host; // what lbm_particles_get reads, where it does not fit lbm_channel::small
};

namespace {

// Final sums of per-block partials of one quantity each: out[c] = the sum of
// part[c*rows + i] in increasing i from 0.0, one block per c.  The block
// brings the partials (at most RED_BLOCKS) into LDS together, so the one
// thread that must add them in order waits for an addition, not for a load
// from memory, per partial (2 048 partials: about 160 us before).
__global__ void __launch_bounds__(256) k_sum_ordered(const double *__restrict__ part, uint32_t rows, double *out)
{
    __shared__ double v[RED_BLOCKS];
    const double *p = part + (uint64_t)blockIdx.x * rows;
    for (uint32_t i = threadIdx.x; i < rows; i += 256)
        v[i] = p[i];
    __syncthreads();
    if (threadIdx.x != 0)
        return;
    double s = 0.0;
#pragma unroll 8
    for (uint32_t i = 0; i < rows; i++)
        s += v[i];
    out[blockIdx.x] = s;
}

// Final sums of the plane sums' partials: out[j] = sum_i part[i*width + j],
// in a fixed order: SUM_ROWS strided sums a column, then those in order.  One
// thread per column waited for each of the 512 loads in turn (143 us for 12
// x 192 columns; 8 us now).
constexpr int SUM_COLS = 64, SUM_ROWS = 16;
__global__ void __launch_bounds__(SUM_COLS *SUM_ROWS)
k_sum_columns(const double *__restrict__ part, uint32_t rows, uint32_t width, double *out, double *acc)
{
    __shared__ double sums[SUM_ROWS][SUM_COLS];
    const uint32_t c = threadIdx.x % SUM_COLS, q = threadIdx.x / SUM_COLS;
    const uint32_t j = blockIdx.x * SUM_COLS + c;
    double s = 0.0;
    if (j < width) {
#pragma unroll 8
        for (uint32_t i = q; i < rows; i += SUM_ROWS)
            s += part[(uint64_t)i * width + j];
    }
    sums[q][c] = s;
    __syncthreads();
    if (q != 0 || j >= width)
        return;
#pragma unroll
    for (int k = 1; k < SUM_ROWS; k++)
        s += sums[k][c];
    out[j] = s;
    if (acc)
        acc[j] += s;
}

// rhoupdat's maximum over its slots into *out (host memory the device can
// write), and the slots back to zero for the next call.  stop, when given, is
// set to whether the maximum is at most eps, and stays set unless first.
__global__ void __launch_bounds__(ERR_SLOTS) k_err_final(unsigned long long *slots, unsigned long long *out,
                                                         unsigned long long *stop, double eps, int first)
{
    static_assert(ERR_SLOTS == 64, "one wave");
    unsigned long long u = slots[threadIdx.x * ERR_STRIDE];
    slots[threadIdx.x * ERR_STRIDE] = 0;
    for (int o = 32; o > 0; o >>= 1) {
        const unsigned long long v = (unsigned long long)__shfl_xor((long long)u, o);
        u = v > u ? v : u;
    }
    if (threadIdx.x == 0) {
        *out = u;
        if (stop) {
            const bool end = __longlong_as_double((long long)u) <= eps;
            if (first || end)
                *stop = end;
        }
    }
}

__global__ void k_sub_scalar(double *__restrict__ a, uint64_t n, double v)
{
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n)
        a[i] = a[i] - v;
}

__global__ void k_fill(double *__restrict__ a, uint64_t n, double v)
{
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n)
        a[i] = v;
}

int dispatch_err(hipError_t e, const char *what)
{
    if (e != hipSuccess)
        return fail(LBM_ERR_HIP, "%s launch failed: %s", what, hipGetErrorString(e));
    return LBM_OK;
}

#define PREC_CALL(h, fn, ...)                                                                   \
    ((h)->prec == LBM_FP64   ? Launch<0>::fn(__VA_ARGS__)                                       \
     : (h)->prec == LBM_FP32 ? Launch<1>::fn(__VA_ARGS__)                                       \
     : (h)->prec == LBM_FP16 ? Launch<2>::fn(__VA_ARGS__)                                       \
                             : Launch<3>::fn(__VA_ARGS__))

RatesD rates_of(const lbm_channel *h)
{
    const lbm_config &c = h->cfg;
    RatesD r;
    r.s1 = c.s1;
    r.s2 = c.s2;
    r.s4 = c.s4;
    r.s9 = c.s9;
    r.s10 = c.s10;
    r.s13 = c.s13;
    r.s16 = c.s16;
    r.omegepsl = c.omegepsl;
    r.omegepslj = c.omegepslj;
    r.omegxx = c.omegxx;
    r.fx = h->fc.fx;
    r.fy = h->fc.fy;
    r.fz = h->fc.fz;
    return with_f32(r);
}

int ensure_fields(lbm_channel *h)
{
    if (h->mac[0])
        return LBM_OK;
    for (int k = 0; k < 4; k++) {
        hipError_t e = hipMalloc((void **)&h->mac[k], h->g.N * sizeof(double));
        if (e != hipSuccess) {
            for (int j = 0; j < k; j++) {
                (void)hipFree(h->mac[j]);
                h->mac[j] = nullptr;
            }
            return fail(LBM_ERR_NOMEM, "hipMalloc of the macroscopic fields (%zu bytes each) failed: %s",
                        (size_t)(h->g.N * sizeof(double)), hipGetErrorString(e));
        }
        HIP_TRY(hipMemsetAsync(h->mac[k], 0, h->g.N * sizeof(double), h->stream));
    }
    return LBM_OK;
}

// macrovar's arguments for nodes [n0, n0 + count) of lattice `which`; the
// caller sets the outputs.
MacroArgs macro_args(const lbm_channel *h, int which, uint64_t n0, uint64_t count)
{
    MacroArgs a;
    a.g = h->g;
    a.L = h->lat[which];
    a.f = h->fm;
    a.rho_off = h->rho_off;
    a.errbits = nullptr;
    a.n0 = (uint32_t)n0;
    a.count = (uint32_t)count;
    return a;
}

// macrovar of lattice `which` (minus the pending rho offset) into the arrays.
int compute_fields(lbm_channel *h, int which)
{
    int rc = ensure_fields(h);
    if (rc)
        return rc;
    MacroArgs a = macro_args(h, which, 0, h->g.N);
    for (int k = 0; k < 4; k++)
        a.out[k] = h->mac[k];
    rc = dispatch_err(PREC_CALL(h, macro, a, 0, h->stream), "macrovar");
    if (rc || !h->part)
        return rc;
    // macrovar's solid branch (collision.f90:420-459), with the current particle state
    const Part *pt = h->part;
    return dispatch_err(part_solid_fields(pt->pg, pt->ps, h->rho_off, h->mac[0], h->mac[1], h->mac[2], h->mac[3],
                                          h->stream),
                        "macrovar inside particles");
}

// macrovar of the current lattice (with the force arrays as they are now)
// becomes what the fields hold.
void fields_from_cur(lbm_channel *h)
{
    h->ms = FROM_CUR;
    h->fm = h->fc;
}

// Do two force specifications give the same force at every node?
bool same_force(const ForceSpec &a, const ForceSpec &b)
{
    return a.tab == b.tab && a.fx == b.fx && a.fy == b.fy && a.fz == b.fz &&
           (a.tab == nullptr || (a.a == b.a && a.b == b.b && a.c == b.c));
}

// Make the arrays hold what the reference's arrays hold now.
int materialize(lbm_channel *h)
{
    if (h->ms == ARRAYS)
        return LBM_OK;
    const int which = (h->ms == FROM_CUR) ? h->cur : 1 - h->cur;
    if (h->ms == FROM_PREV && !h->have_prev)
        return fail(LBM_ERR_STATE, "internal: previous lattice not available");
    int rc = compute_fields(h, which);
    if (rc)
        return rc;
    h->ms = ARRAYS;
    h->rho_off = 0.0;
    return LBM_OK;
}

// Whether the handle's next step is refused, before anything of it is launched.
int step_check(const lbm_channel *h)
{
    const bool arrays = h->ms != FROM_CUR; // the previous lattice's fields go to the arrays first
    if (h->part && (h->fc.tab || (!arrays && !same_force(h->fm, h->fc))))
        return fail(LBM_ERR_STATE, "collision: particles need a uniform force that macrovar has seen "
                                   "(FORCINGP is not combined with particles)");
    if (h->mlp && (arrays || h->rho_off != 0.0)) // the closure runs with fused fields only
        return fail(LBM_ERR_STATE, "collision: the learned closure needs fields from macrovar");
    return LBM_OK;
}

// One step of the handle.  fused: an iteration of the pre-relaxation, whose
// fields are in the arrays and whose force is uniform, without particles or
// closure; it has no effect once *stop is not 0.
int launch_step(lbm_channel *h, bool fused = false, const unsigned long long *stop = nullptr)
{
    const int refused = step_check(h);
    if (refused)
        return refused;
    StepArgs a;
    a.g = h->g;
    a.src = h->lat[h->cur];
    a.dst = h->lat[1 - h->cur];
    a.rho = h->mac[0];
    a.ux = h->mac[1];
    a.uy = h->mac[2];
    a.uz = h->mac[3];
    a.rho_off = h->rho_off;
    a.r = rates_of(h);
    int mode;
    if (h->ms == FROM_PREV) {
        int rc = materialize(h);
        if (rc)
            return rc;
        a.rho = h->mac[0];
        a.ux = h->mac[1];
        a.uy = h->mac[2];
        a.uz = h->mac[3];
        a.rho_off = 0.0;
    }
    if (h->ms == ARRAYS)
        mode = 2;
    else
        mode = (h->rho_off != 0.0) ? 1 : 0;
    a.inside = nullptr;
    if (h->part) {
        mode |= 4;
        a.inside = h->part->ps.inside;
    }
    a.fc = h->fc;
    a.fm = h->fm;
    // a force that varies over the nodes, or fused fields formed with a force
    // other than the collision's
    if (h->fc.tab || (h->ms != ARRAYS && !same_force(h->fm, h->fc)))
        mode |= 16;
    a.mlp = h->mlp;
    a.inv_ystar = h->mlp_inv_ystar;
    a.yscale = h->mlp_yscale;
    a.runs = h->runs;
    a.w32 = h->w32;
    a.to_kept = h->cur == 0;
    a.rho_out = h->mac[0];
    a.errbits = fused ? h->errbits : nullptr;
    a.stop = stop;
    if (h->mlp)
        mode |= 8;
    int rc = dispatch_err(PREC_CALL(h, step, a, mode, h->stream), "collision");
    if (rc)
        return rc;
    h->cur = 1 - h->cur;
    h->have_prev = true;
    h->fresh = false;
    if (h->ms == FROM_CUR)
        h->ms = FROM_PREV;
    return LBM_OK;
}

// Memory for small results the host reads: pinned, or ordinary where no pinned
// memory is to be had.
void *small_alloc(size_t bytes, bool *pinned)
{
    void *p = nullptr;
    *pinned = hipHostMalloc(&p, bytes, hipHostMallocDefault) == hipSuccess;
    if (*pinned)
        return p;
    (void)hipGetLastError();
    return malloc(bytes);
}

void small_free(void *p, bool pinned)
{
    if (pinned)
        (void)hipHostFree(p);
    else
        free(p);
}

hipError_t small_copy(void *small, bool pinned, const void *src, size_t bytes, hipStream_t s)
{
    const hipError_t e = pinned ? link_copy(small, src, bytes, true, s)
                                : hipMemcpyAsync(small, src, bytes, hipMemcpyDeviceToHost, s);
    return e != hipSuccess ? e : hipStreamSynchronize(s);
}

size_t small_bytes(const lbm_channel *h) { return std::max<size_t>(NPLANE * (size_t)h->g.lx, 64) * sizeof(double); }

int ensure_small(lbm_channel *h)
{
    if (!h->small) {
        h->small = (double *)small_alloc(small_bytes(h), &h->small_pinned);
        if (!h->small)
            return fail(LBM_ERR_NOMEM, "allocation of the result buffer failed");
    }
    return LBM_OK;
}

// Where a reduction stores what the host reads next (at most NPLANE * lx
// doubles, after ensure_small): straight to the pinned buffer, since a copy to
// ordinary memory takes 8-10 us longer, or to device memory without one.
double *results_at(const lbm_channel *h) { return h->small_pinned ? h->small : h->red_out + 2; }

// The n doubles stored there, in h->small.
int results(lbm_channel *h, size_t n)
{
    if (!h->small_pinned)
        HIP_TRY(hipMemcpyAsync(h->small, h->red_out + 2, n * sizeof(double), hipMemcpyDeviceToHost, h->stream));
    HIP_TRY(hipStreamSynchronize(h->stream));
    return LBM_OK;
}

// `bytes` of device memory, at most the buffer's size, into h->small.
int read_small(lbm_channel *h, const void *src, size_t bytes)
{
    const int rc = ensure_small(h);
    if (rc)
        return rc;
    HIP_TRY(small_copy(h->small, h->small_pinned, src, bytes, h->stream));
    return LBM_OK;
}

const int *solid_of(const lbm_channel *h) { return h->part ? h->part->ps.solid : nullptr; }

// Sum of rho over fluid nodes (SRC 0: field array, SRC 1: macrovar of the
// current lattice) and the number of fluid nodes.
int reduce_rho(lbm_channel *h, int src, double *sum, double *count)
{
    SumArgs a;
    a.g = h->g;
    a.L = h->lat[h->cur];
    a.rho = h->mac[0];
    a.solid = solid_of(h);
    a.partials = h->partials;
    uint32_t grid = (uint32_t)std::min<uint64_t>(RED_BLOCKS, (h->g.N + 255) / 256);
    int rc = dispatch_err(PREC_CALL(h, rho_partials, a, src, grid, h->stream), "rho reduction");
    if (rc)
        return rc;
    // partials: sums in [0, grid), counts in [grid, 2*grid)
    rc = ensure_small(h);
    if (rc)
        return rc;
    hipLaunchKernelGGL(k_sum_ordered, dim3(2), dim3(256), 0, h->stream, (const double *)h->partials, grid,
                       results_at(h));
    HIP_TRY(hipGetLastError());
    rc = results(h, 2);
    if (rc)
        return rc;
    *sum = h->small[0];
    *count = h->small[1];
    return LBM_OK;
}

// Plane sums of the current fields into out[0 .. 12*lx) (and the running
// accumulator when acc is set).
int plane_sums(lbm_channel *h, double *out, bool acc)
{
    PlaneArgs a;
    a.g = h->g;
    a.L = h->lat[h->ms == FROM_PREV ? 1 - h->cur : h->cur];
    a.rho = h->mac[0];
    a.ux = h->mac[1];
    a.uy = h->mac[2];
    a.uz = h->mac[3];
    a.f = h->fm;
    a.rho_off = h->rho_off;
    a.solid = solid_of(h);
    a.partials = h->partials + 2 * RED_BLOCKS;
    const uint32_t rows = h->g.ly * h->g.lz;
    const uint32_t chunks = std::min<uint32_t>(PLANE_CHUNKS, rows);
    const int src = (h->ms == ARRAYS) ? 0 : 1;
    int rc = dispatch_err(PREC_CALL(h, plane_partials, a, src, chunks, h->stream), "plane sums");
    if (rc)
        return rc;
    const uint32_t width = NPLANE * h->g.lx;
    hipLaunchKernelGGL(k_sum_columns, dim3((width + SUM_COLS - 1) / SUM_COLS), dim3(SUM_COLS * SUM_ROWS), 0, h->stream, a.partials, chunks, width,
                       out, acc ? h->stat_acc : (double *)nullptr);
    HIP_TRY(hipGetLastError());
    return LBM_OK;
}

// Plane sums of the 2x2x2 box-filtered fields of the current populations
// into red_out[2 .. 2 + 12*lx/2) and the filtered running accumulator.
int filtered_plane_sums(lbm_channel *h)
{
    PlaneArgs a;
    a.g = h->g;
    a.L = h->lat[h->ms == FROM_PREV ? 1 - h->cur : h->cur];
    a.rho = a.ux = a.uy = a.uz = nullptr;
    a.f = h->fm;
    a.rho_off = h->rho_off;
    a.solid = nullptr;
    a.partials = h->partials + 2 * RED_BLOCKS;
    const uint32_t rows = (h->g.ly / 2) * (h->g.lz / 2);
    const uint32_t chunks = std::min<uint32_t>(PLANE_CHUNKS, rows);
    int rc = dispatch_err(PREC_CALL(h, filtered_plane_partials, a, chunks, h->stream), "filtered plane sums");
    if (rc)
        return rc;
    const uint32_t width = NPLANE * (h->g.lx / 2);
    hipLaunchKernelGGL(k_sum_columns, dim3((width + SUM_COLS - 1) / SUM_COLS), dim3(SUM_COLS * SUM_ROWS), 0, h->stream, a.partials, chunks, width,
                       h->red_out + 2, h->fstat_acc);
    HIP_TRY(hipGetLastError());
    return LBM_OK;
}

// Columns of saveload.f90:1430-1492 from plane sums s[q*lx + i] of a grid
// with lx planes of plane_nodes nodes; the fluid-node count of plane i is
// s[11*lx + i] (per sample), nsamp the number of accumulated samples.
void stat_columns(uint32_t lx, double plane_nodes, const double *s, double nsamp, double ustar, double ystar,
                  double *out)
{
    const double us2 = ustar * ustar, us4 = us2 * us2;
    for (uint32_t i = 0; i < lx; i++) {
        const double *c = s + i;
        const double nf = c[11 * lx] > 0.0 ? c[11 * lx] : 1.0;
        double vx = c[0 * lx] / nf / ustar, vy = c[1 * lx] / nf / ustar, vz = c[2 * lx] / nf / ustar;
        double sxz = c[3 * lx] / nf / us2 - vx * vz;
        double sxy = c[4 * lx] / nf / us2 - vx * vy;
        double syz = c[5 * lx] / nf / us2 - vy * vz;
        double xx = c[6 * lx] / nf / us2 - vx * vx;
        double yy = c[7 * lx] / nf / us2 - vy * vy;
        double zz = c[8 * lx] / nf / us2 - vz * vz;
        double pr = c[9 * lx] / nf / us2;
        double p2 = c[10 * lx] / nf / us4 - pr * pr;
        const double volf = c[11 * lx] / nsamp / plane_nodes;
        double yplus = ((double)(i + 1) - 0.5) / ystar;
        if (i + 1 > lx / 2)
            yplus = ((double)(lx - (i + 1)) + 0.5) / ystar;
        double *o = out + 15 * (size_t)i;
        o[0] = (double)(i + 1) - 0.5;
        o[1] = yplus;
        o[2] = vx;
        o[3] = vy;
        o[4] = vz;
        o[5] = xx;
        o[6] = yy;
        o[7] = zz;
        o[8] = sxz;
        o[9] = sxy;
        o[10] = syz;
        o[11] = pr;
        o[12] = p2;
        o[13] = volf;
        o[14] = 1.0 - volf;
    }
}

bool same(double a, double b) { return a == b; }

} // namespace

extern "C" {

const char *lbm_last_error(void) { return g_err; }

int lbm_create(const lbm_config *cfg, lbm_channel **out)
{
    g_err[0] = 0;
    if (!cfg || !out)
        return fail(LBM_ERR_ARG, "lbm_create: null argument");
    *out = nullptr;
    const lbm_config &c = *cfg;
    if (c.lx < 2 || c.ly < 1 || c.lz < 1)
        return fail(LBM_ERR_ARG, "lbm_create: grid %d x %d x %d: need lx >= 2, ly >= 1, lz >= 1", c.lx, c.ly, c.lz);
    const uint64_t N = (uint64_t)c.lx * c.ly * c.lz;
    if (N >= (1ull << 31))
        return fail(LBM_ERR_ARG, "lbm_create: %llu nodes exceed the 2^31 per-device limit of 32-bit node indices",
                    (unsigned long long)N);
    if (c.precision < LBM_FP64 || c.precision > LBM_FP16C)
        return fail(LBM_ERR_ARG, "lbm_create: unknown precision %d", c.precision);
    if (c.reserved != 0)
        return fail(LBM_ERR_ARG, "lbm_create: reserved field must be 0");
    // structural constants are compiled into the kernels (para.f90:143-174)
    struct {
        const char *name;
        double got, want;
    } chk[] = {{"coef1", c.coef1, -(2.0 / 3.0)}, {"coef2", c.coef2, -11.0},        {"coef3", c.coef3, 8.0},
               {"coef4", c.coef4, -4.0},         {"coef5", c.coef5, 2.0},          {"coef3i", c.coef3i, 1.0 / 8.0},
               {"coef4i", c.coef4i, 1.0 / -4.0}, {"val8", c.val8, 12.0},           {"val1i", c.val1i, 1.0 / 19.0},
               {"val2i", c.val2i, 1.0 / 2394.0}, {"val3i", c.val3i, 1.0 / 252.0},  {"val4i", c.val4i, 1.0 / 10.0},
               {"val5i", c.val5i, 1.0 / 40.0},   {"val6i", c.val6i, 1.0 / 36.0},   {"val7i", c.val7i, 1.0 / 72.0},
               {"val8i", c.val8i, 1.0 / 12.0},   {"val9i", c.val9i, 1.0 / 24.0},   {"ww0", c.ww0, 1.0 / 3.0},
               {"ww1", c.ww1, 1.0 / 18.0},       {"ww2", c.ww2, 1.0 / 36.0}};
    for (auto &k : chk)
        if (!same(k.got, k.want))
            return fail(LBM_ERR_ARG, "lbm_create: %s = %.17g differs from Channel-Flow/para.f90's %.17g", k.name,
                        k.got, k.want);

    int ndev = 0;
    HIP_TRY(hipGetDeviceCount(&ndev));
    if (c.device < 0 || c.device >= ndev)
        return fail(LBM_ERR_ARG, "lbm_create: device %d not present (%d devices)", c.device, ndev);
    if (c.device >= MAX_DEVICES)
        return fail(LBM_ERR_ARG, "lbm_create: device %d beyond the library's %d-device table", c.device, MAX_DEVICES);
    HIP_TRY(hipSetDevice(c.device));
    {
        // device address of this GPU's copy of `scratch`, once per device
        std::lock_guard<std::mutex> lock(g_scratch_mu);
        if (!g_scratch_ptr[c.device]) {
            void *p = nullptr;
            HIP_TRY(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
            if (!p)
                return fail(LBM_ERR_HIP, "lbm_create: hipGetSymbolAddress(scratch) gave a null address");
            g_scratch_ptr[c.device] = (double *)p;
        }
    }

    lbm_channel *h = new lbm_channel();
    memset(h, 0, sizeof(*h));
    host_pool().retain();
    h->cfg = c;
    h->prec = c.precision;
    h->elem = c.precision == LBM_FP64 ? 8 : (c.precision == LBM_FP32 ? 4 : 2);
    h->g.lx = c.lx;
    h->g.ly = c.ly;
    h->g.lz = c.lz;
    h->g.plane = (uint32_t)c.lx * c.ly;
    h->g.N = N;
    h->g.S = padded_stride(N, h->elem);
    h->g.dlx = make_fastdiv(c.lx);
    h->g.dly = make_fastdiv(c.ly);
    h->g.remap = 0;
    {
        // LBM_STEP_KERNEL=runs selects two nodes per thread (measured slower on
        // the 192x768x384 channel: 64.6 % vs 69.2 % of HBM in FP64)
        const char *k = getenv("LBM_STEP_KERNEL");
        h->runs = (k && strcmp(k, "runs") == 0) ? 1 : 0;
        // LBM_STEP_W32=0: 2-byte storage, the FP32 closure and FP32 steps of
        // lattices beyond the last-level cache address their pulls with
        // 64-bit arithmetic even where 32-bit offsets would do;
        // LBM_STEP_W32=adjacent: 2-byte storage takes 32-bit
        // offsets between adjacent rows only, the form lattices above 2^29
        // nodes use (the same values; for comparing the forms)
        const char *w = getenv("LBM_STEP_W32");
        h->w32 = (w && strcmp(w, "0") == 0) ? 0 : (w && strcmp(w, "adjacent") == 0) ? 2 : 1;
        // two-step blocked sweep (blocked.h, block_choice): chunks of K slabs
        // whose ring of K + 2 slabs stays within BLOCK_RING_BYTES, along the
        // axis whose chunk holds more nodes.  Below BLOCK_MIN_SLABS whole
        // slabs measured slower than single steps (the 2048x1024x512
        // channel's 40 MB y slabs allow two: 33 900 against 38 200 MLUPS), so
        // the slabs are then cut into row windows (there: four of 256 rows,
        // 20 to a chunk, 42 100-42 200 MLUPS in FP32).  On
        // the 192x768x384 channel this picks 11.2 MB slabs, 18 to a chunk, in
        // both FP64 (y: 20 650-20 700 MLUPS against 20 000-20 090 for z
        // slabs, 8 to a chunk) and FP32 (z: about 42 000).
        // LBM_BLOCK_AXIS=z|y sets the axis, LBM_BLOCK_PLANES=K the chunk (0:
        // off), LBM_BLOCK_ROWS=W row windows of W rows (0: whole slabs).  Not
        // by default for 2-byte storage, whose step is bound by arithmetic
        // (FP16: measured 66 300 MLUPS blocked, 32 to a chunk, against 72 000
        // single-step).
        // Rows that are not whole cache lines are swept along z: z slabs are
        // contiguous, so their waves can start on lines (BlockArgs::res).
        const char *axis = getenv("LBM_BLOCK_AXIS");
        if (!axis && c.lx * h->elem % 128 != 0 && (uint64_t)c.lx * c.ly * 19 * h->elem * (BLOCK_MIN_SLABS + 2) <=
                                                      (uint64_t)BLOCK_RING_BYTES)
            axis = "z";
        const BlockChoice bc =
            block_choice(h->g, h->elem, h->elem != 2, BLOCK_RING_BYTES, BLOCK_MIN_SLABS, axis,
                         getenv("LBM_BLOCK_PLANES"), getenv("LBM_BLOCK_ROWS"));
        if (bc.bad) {
            (void)lbm_destroy(h);
            return fail(LBM_ERR_ARG, "lbm_create: invalid value of %s", bc.bad);
        }
        h->baxis = bc.axis;
        h->bK = bc.K;
        h->bW = bc.W;
        // small lattices and chunks are faster in single steps; setting the
        // sweep's variables asks for the sweep at any size
        const uint64_t chunk_rows = bc.W ? bc.W : block_geom(h->g, bc.axis).nr;
        h->bskip = (N * 19 * h->elem <= BLOCK_MIN_LATTICE_BYTES ||
                    bc.K * chunk_rows * c.lx * 19 * h->elem < BLOCK_MIN_CHUNK_BYTES) &&
                   !getenv("LBM_BLOCK_AXIS") && !getenv("LBM_BLOCK_PLANES") && !getenv("LBM_BLOCK_ROWS");
        // Pairs under a force evaluated per node run as sweeps too
        // (LBM_BLOCK_FORCED=0: as single steps).  With both steps' forces
        // from one set of factors (node_forces) that is the faster form: us
        // per step on 96x384x192, FP64 361 against 394 for single steps, FP32
        // 191 / 199; on 192x768x384 2 869 / 3 081 and 1 403 / 1 607.
        const char *kf = getenv("LBM_BLOCK_FORCED");
        h->bforced = (kf && strcmp(kf, "0") == 0) ? 0 : 1;
        // LBM_DEFER=0: collision_MRT launches at once (no per-call pairing)
        const char *kd = getenv("LBM_DEFER");
        if (kd && strcmp(kd, "0") != 0 && strcmp(kd, "1") != 0) {
            (void)lbm_destroy(h);
            return fail(LBM_ERR_ARG, "lbm_create: invalid value of LBM_DEFER (0 or 1)");
        }
        h->defer = (kd && strcmp(kd, "0") == 0) ? 0 : 1;
        // LBM_PART_STREAMS=1|2: lbm_run_particles on so many streams (default:
        // by the lattice's size)
        const char *kp = getenv("LBM_PART_STREAMS");
        if (kp && strcmp(kp, "1") != 0 && strcmp(kp, "2") != 0) {
            (void)lbm_destroy(h);
            return fail(LBM_ERR_ARG, "lbm_create: invalid value of LBM_PART_STREAMS (1 or 2)");
        }
        h->pstreams = kp ? kp[0] - '0' : 0;
    }
    fields_from_cur(h);
    h->fresh = true;

    auto cleanup = [&](int code) {
        lbm_destroy(h);
        return code;
    };
    hipError_t e = hipStreamCreateWithFlags(&h->stream, hipStreamNonBlocking);
    if (e != hipSuccess)
        return cleanup(fail(LBM_ERR_HIP, "hipStreamCreate failed: %s", hipGetErrorString(e)));
    const size_t lat_bytes = (size_t)h->g.S * 19 * h->elem;
    for (int k = 0; k < 2; k++) {
        e = hipMalloc(&h->lat[k], lat_bytes);
        if (e != hipSuccess)
            return cleanup(fail(LBM_ERR_NOMEM, "hipMalloc of lattice %d (%zu bytes) failed: %s", k, lat_bytes,
                                hipGetErrorString(e)));
        e = hipMemsetAsync(h->lat[k], 0, lat_bytes, h->stream);
        if (e != hipSuccess)
            return cleanup(fail(LBM_ERR_HIP, "hipMemsetAsync failed: %s", hipGetErrorString(e)));
    }
    const size_t part = 2 * RED_BLOCKS + (size_t)PLANE_CHUNKS * NPLANE * c.lx;
    if (hipMalloc((void **)&h->partials, part * sizeof(double)) != hipSuccess ||
        hipMalloc((void **)&h->red_out, (2 + NPLANE * (size_t)c.lx) * sizeof(double)) != hipSuccess ||
        hipMalloc((void **)&h->stat_acc, NPLANE * (size_t)c.lx * sizeof(double)) != hipSuccess ||
        hipMalloc((void **)&h->errbits, ERR_BYTES) != hipSuccess)
        return cleanup(fail(LBM_ERR_NOMEM, "hipMalloc of reduction scratch failed"));
    e = hipMemsetAsync(h->stat_acc, 0, NPLANE * (size_t)c.lx * sizeof(double), h->stream);
    if (e == hipSuccess)
        e = hipMemsetAsync(h->errbits, 0, ERR_SLOTS * ERR_STRIDE * sizeof(unsigned long long), h->stream);
    if (e == hipSuccess)
        e = hipEventCreate(&h->ev[0]);
    if (e == hipSuccess)
        e = hipEventCreate(&h->ev[1]);
    if (e == hipSuccess)
        e = hipStreamSynchronize(h->stream);
    if (e != hipSuccess)
        return cleanup(fail(LBM_ERR_HIP, "lbm_create setup failed: %s", hipGetErrorString(e)));
    *out = h;
    return LBM_OK;
}

int lbm_destroy(lbm_channel *h)
{
    if (!h)
        return LBM_OK;
    (void)hipSetDevice(h->cfg.device);
    if (h->stream)
        (void)hipStreamSynchronize(h->stream);
    if (h->pstream) // particle work an error return left unjoined
        (void)hipStreamSynchronize(h->pstream);
    for (int k = 0; k < 2; k++)
        if (h->lat[k])
            (void)hipFree(h->lat[k]);
    for (int k = 0; k < 4; k++)
        if (h->mac[k])
            (void)hipFree(h->mac[k]);
    if (h->partials)
        (void)hipFree(h->partials);
    if (h->red_out)
        (void)hipFree(h->red_out);
    if (h->stat_acc)
        (void)hipFree(h->stat_acc);
    if (h->fstat_acc)
        (void)hipFree(h->fstat_acc);
    if (h->errbits)
        (void)hipFree(h->errbits);
    if (h->errout)
        (void)hipHostFree(h->errout);
    small_free(h->small, h->small_pinned);
    if (h->stage)
        (void)hipFree(h->stage);
    if (h->part) {
        for (void *p : h->part->allocs)
            (void)hipFree(p);
        delete h->part;
    }
    if (h->mlp)
        (void)hipFree(h->mlp);
    if (h->ftab)
        (void)hipFree(h->ftab);
    if (h->bring)
        (void)hipFree(h->bring);
    if (h->bhead)
        (void)hipFree(h->bhead);
    for (hipEvent_t e : h->pev)
        if (e)
            (void)hipEventDestroy(e);
    if (h->pstream)
        (void)hipStreamDestroy(h->pstream);
    if (h->ev[0])
        (void)hipEventDestroy(h->ev[0]);
    if (h->ev[1])
        (void)hipEventDestroy(h->ev[1]);
    host_pool().release(); // before the handle's own stream goes
    if (h->stream)
        (void)hipStreamDestroy(h->stream);
    delete h;
    return LBM_OK;
}

// Launches the collisions lbm_collision_mrt deferred, as single steps, and
// leaves the state the calls one by one would have left: the first step, the
// fields of a macrovar that followed it, the second step (whose macrovar has
// not come, or the pair would have run).
static int flush_pending(lbm_channel *h)
{
    const int n = h->pend;
    if (n == 0)
        return LBM_OK;
    const bool mac = h->pend_mac;
    h->pend = 0;
    h->pend_mac = false;
    int rc = launch_step(h);
    if (rc)
        return rc;
    if (n == 1 && !mac)
        return LBM_OK; // fields FROM_PREV, as launch_step left them
    fields_from_cur(h);
    h->rho_off = 0.0;
    return n == 2 ? launch_step(h) : LBM_OK;
}

// Entry with no deferred work flushed: lbm_collision_mrt and lbm_macrovar.
#define CHECK_H_KEEP(h)                                                  \
    do {                                                                 \
        if (!(h))                                                        \
            return fail(LBM_ERR_ARG, "%s: null handle", __func__);       \
        g_err[0] = 0;                                                    \
        HIP_TRY(hipSetDevice((h)->cfg.device));                          \
    } while (0)

// Every other entry point first launches deferred collisions, so it sees the
// state the calls one by one leave.
#define CHECK_H(h)                                                       \
    do {                                                                 \
        CHECK_H_KEEP(h);                                                 \
        const int frc_ = flush_pending(h);                               \
        if (frc_)                                                        \
            return frc_;                                                 \
    } while (0)

static int ensure_stage(lbm_channel *h)
{
    if (h->stage)
        return LBM_OK;
    hipError_t e = hipMalloc((void **)&h->stage, STAGE_BYTES);
    if (e != hipSuccess)
        return fail(LBM_ERR_NOMEM, "hipMalloc of the copy staging buffer failed: %s", hipGetErrorString(e));
    return LBM_OK;
}

extern "C++" {
namespace {

// Nodes [0, N) in slices of at most slice_bytes of node_bytes each.
struct NodeSlices {
    uint64_t N, per;
    size_t node_bytes;
    NodeSlices(uint64_t n, size_t nb, size_t slice_bytes) : N(n), per(slice_bytes / nb / 256 * 256), node_bytes(nb) {}
    size_t count() const { return (size_t)((N + per - 1) / per); }
    uint64_t first(size_t k) const { return k * per; }
    uint64_t nodes(size_t k) const { return std::min<uint64_t>(per, N - k * per); }
    size_t bytes(size_t k) const { return (size_t)nodes(k) * node_bytes; }
};

// Per-node values made on the device slice by slice into nout host arrays of
// node_bytes each (null ones are skipped): launch(first, nodes, dst, step,
// stream) writes those of array j to dst + j * step bytes, j counting the
// arrays that are not null.  The kernels store straight into the pinned slots, unless
// their stores are scattered (`staged`: through device slices).
template <class Launch>
int nodes_to_host(lbm_channel *h, void *const *out, int nout, size_t node_bytes, bool staged, const char *what,
                  Launch launch)
{
    char *host[4];
    int m = 0;
    bool known = false;
    for (int j = 0; j < nout; j++)
        if (out[j])
            host[m++] = (char *)out[j];
    const hipStream_t s = h->stream;
    const size_t total = h->g.N * node_bytes * m;
    // the runtime takes several pinned arrays one after another, 8 us each: up
    // to 1 MiB for each after the first the slots are faster (us through the
    // slots / by the runtime, 0.8 MB of fields 45 / 60, 2.1 MB 83 / 88, 5.2 MB
    // 205 / 151)
    for (int j = 0; j < m && total >= HOST_MIN; j++) {
        const hipMemoryType t = array_type(host[j]);
        known = known || (t == hipMemoryTypeHost ? total >= (size_t)(m - 1) << 20 : t != hipMemoryTypeUnregistered);
    }
    const bool sliced = total >= HOST_MIN && !known;
    if (sliced)
        HIP_TRY(hipStreamSynchronize(s));
    HostPool &pool = host_pool();
    const int workers = host_workers(total, true);
    std::unique_lock<std::mutex> lock(pool.mu, std::defer_lock);
    hipError_t e = hipSuccess;
    const bool pooled = sliced && lock.try_lock() && pool.ready(h->cfg.device, workers);
    if (staged || !pooled) {
        const int rc = ensure_stage(h);
        if (rc)
            return rc;
    }
    if (pooled) {
        const NodeSlices sl(h->g.N, node_bytes * m, host_slice(total, true));
        const size_t step = sl.per * node_bytes;
        e = host_slices_out(
            pool, h->cfg.device, s, sl.count(), workers,
            [&](size_t k, int slot, char *pinned, hipStream_t on) {
                char *dev = staged ? h->stage + slot * HOST_SLICE : pinned;
                const hipError_t le = launch(sl.first(k), sl.nodes(k), dev, step, on);
                return le != hipSuccess || !staged ? le : link_copy(pinned, dev, sl.bytes(k), true, on);
            },
            [&](size_t k, const char *pinned) {
                for (int j = 0; j < m; j++)
                    memcpy(host[j] + sl.first(k) * node_bytes, pinned + j * step, sl.nodes(k) * node_bytes);
            });
    } else {
        const NodeSlices sl(h->g.N, node_bytes * m, STAGE_BYTES);
        const size_t step = sl.per * node_bytes;
        for (size_t k = 0; k < sl.count() && e == hipSuccess; k++) {
            e = launch(sl.first(k), sl.nodes(k), h->stage, step, s);
            for (int j = 0; j < m && e == hipSuccess; j++)
                e = hipMemcpyAsync(host[j] + sl.first(k) * node_bytes, h->stage + j * step, sl.nodes(k) * node_bytes,
                                   hipMemcpyDeviceToHost, s);
            if (e == hipSuccess)
                e = hipStreamSynchronize(s);
        }
    }
    if (e != hipSuccess)
        return fail(LBM_ERR_HIP, "%s: %s", what, hipGetErrorString(e));
    return LBM_OK;
}

// The host array `in` to the device slice by slice, launch consuming each,
// straight from the pinned slot.
template <class Launch>
int nodes_from_host(lbm_channel *h, const void *in, size_t node_bytes, const char *what, Launch launch)
{
    const char *const host = (const char *)in;
    const hipStream_t s = h->stream;
    const size_t total = h->g.N * node_bytes;
    const bool sliced = total >= HOST_MIN && !runtime_array(host);
    if (sliced)
        HIP_TRY(hipStreamSynchronize(s));
    HostPool &pool = host_pool();
    const int workers = host_workers(total, false);
    std::unique_lock<std::mutex> lock(pool.mu, std::defer_lock);
    hipError_t e = hipSuccess;
    if (sliced && lock.try_lock() && pool.ready(h->cfg.device, workers)) {
        const NodeSlices sl(h->g.N, node_bytes, host_slice(total, false));
        e = host_slices_in(
            pool, h->cfg.device, s, sl.count(), workers,
            [&](size_t k, char *pinned) { memcpy(pinned, host + sl.first(k) * node_bytes, sl.bytes(k)); },
            [&](size_t k, int, const char *pinned, hipStream_t on) {
                return launch(sl.first(k), sl.nodes(k), (char *)pinned, on);
            });
    } else {
        const int rc = ensure_stage(h);
        if (rc)
            return rc;
        const NodeSlices sl(h->g.N, node_bytes, STAGE_BYTES);
        for (size_t k = 0; k < sl.count() && e == hipSuccess; k++) {
            e = hipMemcpyAsync(h->stage, host + sl.first(k) * node_bytes, sl.bytes(k), hipMemcpyHostToDevice, s);
            if (e == hipSuccess)
                e = launch(sl.first(k), sl.nodes(k), h->stage, s);
        }
        if (e == hipSuccess)
            e = hipStreamSynchronize(s);
    }
    if (e != hipSuccess)
        return fail(LBM_ERR_HIP, "%s: %s", what, hipGetErrorString(e));
    return LBM_OK;
}

// Whole arrays between host and device; null host pointers are skipped.
int copy_parts(lbm_channel *h, const HostPart *parts, int n, bool down, const char *what)
{
    const hipError_t e = host_copy(h->cfg.device, h->stream, parts, n, down);
    if (e != hipSuccess)
        return fail(LBM_ERR_HIP, "%s: copy failed: %s", what, hipGetErrorString(e));
    return LBM_OK;
}

} // namespace
} // extern "C++"

int lbm_upload_f(lbm_channel *h, const double *f)
{
    CHECK_H(h);
    if (!f)
        return fail(LBM_ERR_ARG, "lbm_upload_f: null f");
    // the reference's arrays keep their values when f is replaced
    if (!h->fresh && h->ms != ARRAYS) {
        const int rc = materialize(h);
        if (rc)
            return rc;
    }
    const int rc = nodes_from_host(h, f, 19 * sizeof(double), "lbm_upload_f", [h](uint64_t n0, uint64_t cnt, char *dev, hipStream_t on) {
        CopyArgs a;
        a.g = h->g;
        a.L = h->lat[h->cur];
        a.aos = (double *)dev;
        a.n0 = n0;
        a.count = cnt;
        return PREC_CALL(h, scatter, a, on);
    });
    if (rc)
        return rc;
    h->have_prev = false;
    return LBM_OK;
}

int lbm_download_f(lbm_channel *h, double *f)
{
    CHECK_H(h);
    if (!f)
        return fail(LBM_ERR_ARG, "lbm_download_f: null f");
    void *const out[1] = {f};
    return nodes_to_host(h, out, 1, 19 * sizeof(double), false, "lbm_download_f",
                         [h](uint64_t n0, uint64_t cnt, char *dev, size_t, hipStream_t on) {
        CopyArgs a;
        a.g = h->g;
        a.L = h->lat[h->cur];
        a.aos = (double *)dev;
        a.n0 = n0;
        a.count = cnt;
        return PREC_CALL(h, gather, a, on);
    });
}

int lbm_set_force(lbm_channel *h, double fx, double fy, double fz)
{
    CHECK_H(h);
    // the fields keep the force they were formed with (fm) until the next
    // macrovar; a fresh handle has formed none yet
    h->fc.fx = fx;
    h->fc.fy = fy;
    h->fc.fz = fz;
    h->fc.tab = nullptr;
    h->fc.a = h->fc.b = h->fc.c = 0.0;
    if (h->fresh)
        h->fm = h->fc;
    return LBM_OK;
}

int lbm_forcingp(lbm_channel *h, int istep, double force_in_y)
{
    CHECK_H(h);
    if (h->part)
        return fail(LBM_ERR_STATE, "lbm_forcingp: not for particle-laden channels (Channel-Flow/main.f90:148)");
    const uint32_t lx = h->g.lx, ly = h->g.ly, lz = h->g.lz;
    const double pi2 = 2.0 * (4.0 * atan(1.0)); // var_inc.f90:71-72
    const double beta9 = 3.0, gamma9 = 2.0, phase9 = 0.25, Tpd = 2000.;
    const int ixs0 = 2;
    const int ihh = (int)(lx / 2) / 2; // lxh/2, var_inc.f90:53
    if (!h->ftab) {
        // factors of one coordinate each (collision.f90:561-599, one rank);
        // computed with the C library's sin and cos, as the oracle does
        std::vector<double> t(3 * (size_t)lx + 4 * (size_t)ly + 2 * (size_t)lz, 0.0);
        for (int band = 1; band <= 2; band++) {
            const int ixs = band == 1 ? ixs0 : (int)lx - ixs0 - ihh; // the second band is written last
            for (int i = 1; i <= ihh; i++) {
                const double x9 = pi2 * ((double)i - 0.5) / (double)ihh;
                double *xt = &t[3 * (size_t)(i + ixs - 1)];
                xt[0] = (double)band;
                xt[1] = 1. - cos(x9);
                xt[2] = sin(x9);
            }
        }
        for (uint32_t j = 1; j <= ly; j++) {
            const double y1 = pi2 * ((double)j - 0.5) / (double)ly;
            const double y2 = pi2 * (((double)j - 0.5) / (double)ly + phase9);
            double *yt = &t[3 * (size_t)lx + 4 * (size_t)(j - 1)];
            yt[0] = cos(beta9 * y1);
            yt[1] = sin(beta9 * y1);
            yt[2] = cos(beta9 * y2);
            yt[3] = sin(beta9 * y2);
        }
        for (uint32_t k = 1; k <= lz; k++) {
            const double z9 = pi2 * ((double)k - 0.5) / (double)lz;
            double *zt = &t[3 * (size_t)lx + 4 * (size_t)ly + 2 * (size_t)(k - 1)];
            zt[0] = cos(gamma9 * z9);
            zt[1] = sin(gamma9 * z9);
        }
        hipError_t e = hipMalloc((void **)&h->ftab, t.size() * sizeof(double));
        if (e != hipSuccess)
            return fail(LBM_ERR_NOMEM, "hipMalloc of the FORCINGP tables failed: %s", hipGetErrorString(e));
        HIP_TRY(hipMemcpyAsync(h->ftab, t.data(), t.size() * sizeof(double), hipMemcpyHostToDevice, h->stream));
        HIP_TRY(hipStreamSynchronize(h->stream));
    }
    // collision.f90:541 and the amplitude factors of :571-576
    const double Amp0 = 40.00 * beta9 / (double)ly * sin(pi2 * (double)istep / Tpd);
    h->fc.fx = 0.0;
    h->fc.fy = force_in_y;
    h->fc.fz = 0.0;
    h->fc.tab = h->ftab;
    h->fc.a = force_in_y * 0.5 * Amp0 * (double)ihh;
    h->fc.b = Amp0 * (double)ly / beta9;
    h->fc.c = force_in_y * 0.5 * Amp0 * (double)lz / gamma9;
    if (h->fresh)
        h->fm = h->fc;
    return LBM_OK;
}

int lbm_set_macros(lbm_channel *h, const double *rho, const double *ux, const double *uy, const double *uz)
{
    CHECK_H(h);
    int rc = materialize(h);
    if (rc)
        return rc;
    const double *src[4] = {rho, ux, uy, uz};
    HostPart parts[4];
    for (int k = 0; k < 4; k++)
        parts[k] = HostPart{const_cast<double *>(src[k]), h->mac[k], h->g.N * sizeof(double)};
    rc = copy_parts(h, parts, 4, false, "lbm_set_macros");
    if (rc)
        return rc;
    h->fresh = false;
    return LBM_OK;
}

namespace {

constexpr int SEP_MAX_TERMS = 64;
struct SepTerms {
    int n;
    int comp[SEP_MAX_TERMS];
};

// rho = 0 and u_c = sum over the terms k of component c of
// planes[k][row] * profiles[k][ix] (row = iy + ly*iz), in increasing k from 0.
__global__ void k_separable(Geom g, SepTerms t, const double *__restrict__ planes,
                            const double *__restrict__ profiles, double *rho, double *ux, double *uy, double *uz)
{
    const uint64_t n = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= g.N)
        return;
    const uint64_t row = n / g.lx, ix = n - row * g.lx;
    const uint64_t rows = g.N / g.lx;
    double u[3] = {0.0, 0.0, 0.0};
    for (int k = 0; k < t.n; k++)
        u[t.comp[k]] = u[t.comp[k]] + planes[(uint64_t)k * rows + row] * profiles[(uint64_t)k * g.lx + ix];
    rho[n] = 0.0;
    ux[n] = u[0];
    uy[n] = u[1];
    uz[n] = u[2];
}

} // namespace

int lbm_set_velocity_separable(lbm_channel *h, int nterms, const int *comp, const double *planes,
                               const double *profiles)
{
    CHECK_H(h);
    if (nterms < 1 || nterms > SEP_MAX_TERMS || !comp || !planes || !profiles)
        return fail(LBM_ERR_ARG, "lbm_set_velocity_separable: need 1 <= nterms <= %d and non-null arrays",
                    SEP_MAX_TERMS);
    SepTerms t;
    t.n = nterms;
    for (int k = 0; k < nterms; k++) {
        if (comp[k] < 0 || comp[k] > 2)
            return fail(LBM_ERR_ARG, "lbm_set_velocity_separable: term %d has component %d (0, 1 or 2)", k, comp[k]);
        t.comp[k] = comp[k];
    }
    int rc = materialize(h);
    if (rc)
        return rc;
    const size_t rows = (size_t)h->g.ly * h->g.lz;
    const size_t pb = (size_t)nterms * rows * sizeof(double), qb = (size_t)nterms * h->g.lx * sizeof(double);
    double *dp = nullptr, *dq = nullptr;
    hipError_t e = hipMalloc((void **)&dp, pb);
    if (e == hipSuccess)
        e = hipMalloc((void **)&dq, qb);
    if (e == hipSuccess)
        e = hipMemcpyAsync(dp, planes, pb, hipMemcpyHostToDevice, h->stream);
    if (e == hipSuccess)
        e = hipMemcpyAsync(dq, profiles, qb, hipMemcpyHostToDevice, h->stream);
    if (e == hipSuccess) {
        hipLaunchKernelGGL(k_separable, dim3((unsigned)((h->g.N + 255) / 256)), dim3(256), 0, h->stream, h->g, t, dp,
                           dq, h->mac[0], h->mac[1], h->mac[2], h->mac[3]);
        e = hipGetLastError();
    }
    if (e == hipSuccess)
        e = hipStreamSynchronize(h->stream);
    if (dp)
        (void)hipFree(dp);
    if (dq)
        (void)hipFree(dq);
    if (e != hipSuccess)
        return fail(LBM_ERR_HIP, "lbm_set_velocity_separable: %s", hipGetErrorString(e));
    h->fresh = false;
    return LBM_OK;
}

int lbm_initpop(lbm_channel *h)
{
    CHECK_H(h);
    int rc = materialize(h);
    if (rc)
        return rc;
    InitArgs a;
    a.g = h->g;
    a.L = h->lat[h->cur];
    a.rho = h->mac[0];
    a.ux = h->mac[1];
    a.uy = h->mac[2];
    a.uz = h->mac[3];
    rc = dispatch_err(PREC_CALL(h, initpop, a, h->stream), "initpop");
    if (rc)
        return rc;
    h->have_prev = false;
    h->fresh = false;
    return LBM_OK;
}

static bool block_ready(const lbm_channel *h);
static int run_pair(lbm_channel *h);

int lbm_collision_mrt(lbm_channel *h)
{
    CHECK_H_KEEP(h);
    // Per-call pairing: a collision that lbm_run could pair is deferred; if
    // macrovar and another collision follow, the two run as one blocked pair
    // at the next macrovar (bitwise the single steps).  Any other call
    // launches what is deferred first.
    if (h->defer && h->pend == 0 && block_ready(h)) {
        h->pend = 1;
        h->pend_mac = false;
        return LBM_OK;
    }
    if (h->pend == 1 && h->pend_mac) {
        h->pend = 2;
        return LBM_OK;
    }
    const int rc = flush_pending(h);
    if (rc)
        return rc;
    return launch_step(h);
}

int lbm_macrovar(lbm_channel *h, double *rho, double *ux, double *uy, double *uz)
{
    CHECK_H_KEEP(h);
    if (h->pend && !rho && !ux && !uy && !uz) {
        if (h->pend == 1) { // fields of the deferred step (again, if twice)
            h->pend_mac = true;
            return LBM_OK;
        }
        h->pend = 0; // collision, macrovar, collision, macrovar: one pair
        h->pend_mac = false;
        return run_pair(h);
    }
    const int frc = flush_pending(h);
    if (frc)
        return frc;
    fields_from_cur(h);
    h->rho_off = 0.0;
    h->fresh = false;
    double *dst[4] = {rho, ux, uy, uz};
    if (!rho && !ux && !uy && !uz)
        return LBM_OK;
    if (h->part) { // nodes inside particles are set in the arrays
        int rc = compute_fields(h, h->cur);
        if (rc)
            return rc;
        HostPart parts[4];
        for (int k = 0; k < 4; k++)
            parts[k] = HostPart{dst[k], h->mac[k], h->g.N * sizeof(double)};
        return copy_parts(h, parts, 4, true, "lbm_macrovar");
    }
    void *const out[4] = {rho, ux, uy, uz};
    return nodes_to_host(h, out, 4, sizeof(double), false, "lbm_macrovar",
                         [h, &dst](uint64_t n0, uint64_t cnt, char *dev, size_t step, hipStream_t on) {
                             MacroArgs a = macro_args(h, h->cur, n0, cnt);
                             for (int k = 0; k < 4; k++) {
                                 a.out[k] = dst[k] ? (double *)dev : nullptr;
                                 dev += dst[k] ? step : 0;
                             }
                             return PREC_CALL(h, macro, a, 0, on);
                         });
}

// Pinned results of rhoupdat: a word for each iteration of lbm_prerelax, whose
// loop prepares and reads them without waiting for the stream, and behind them
// one of lbm_rhoupdat's own, whose kernel may still be queued by then when the
// caller did not ask for the maximum.
constexpr int PRE_ITERS = 64;

// False without pinned memory: rhoupdat then takes its maximum from device
// memory, and lbm_prerelax makes the calls one by one.
static bool ensure_errout(lbm_channel *h)
{
    if (!h->errout &&
        hipHostMalloc((void **)&h->errout, (PRE_ITERS + 1) * sizeof(unsigned long long), hipHostMallocDefault) !=
            hipSuccess) {
        (void)hipGetLastError();
        h->errout = nullptr;
    }
    return h->errout != nullptr;
}

int lbm_rhoupdat(lbm_channel *h, double *rhoerrmax)
{
    CHECK_H(h);
    // u keeps what the arrays hold; rho becomes sum f of the current lattice
    int rc = materialize(h);
    if (rc)
        return rc;
    const bool pinned = ensure_errout(h);
    MacroArgs a = macro_args(h, h->cur, 0, h->g.N);
    a.out[0] = h->mac[0];
    a.errbits = h->errbits;
    rc = dispatch_err(PREC_CALL(h, macro, a, 1, h->stream), "rhoupdat");
    if (rc)
        return rc;
    // the device writes the result where the host reads it: the loop waits for
    // this value every iteration (a copy to ordinary memory and the clearing
    // of the slots before the kernel took 12 us longer)
    unsigned long long *const out = pinned ? h->errout + PRE_ITERS : (unsigned long long *)h->red_out;
    hipLaunchKernelGGL(k_err_final, dim3(1), dim3(ERR_SLOTS), 0, h->stream, h->errbits, out,
                       (unsigned long long *)nullptr, 0.0, 0);
    HIP_TRY(hipGetLastError());
    h->fresh = false;
    if (rhoerrmax) {
        if (!pinned)
            HIP_TRY(hipMemcpyAsync(rhoerrmax, out, sizeof(double), hipMemcpyDeviceToHost, h->stream));
        HIP_TRY(hipStreamSynchronize(h->stream));
        if (pinned)
            memcpy(rhoerrmax, out, sizeof(double));
    }
    return LBM_OK;
}

// Iterations ahead of the last one whose result the host has seen.  The first of
// a call runs alone (`hold`): from initpop's populations it often is the last, as
// the equilibrium's own density changes by nothing, and the three iterations
// after it would read the lattice for nothing (96x384x192, us of a loop of one
// iteration: FP64 1 122, 461 alone, 844 with the calls one by one; FP32 709 / 269
// / 621).  Two iterations with three in vain are still faster than two by calls.
constexpr int PRE_AHEAD = 4;

// The iterations run ahead of the host's test: it reads each maximum from
// pinned memory while later iterations run, and those find the stop word set
// and do nothing.  us per iteration, calls one by one / this loop: FP64
// 16x32x32 21.6 / 7.9, 64x192x96 108 / 69, 96x384x192 655 / 444; FP32 20.4 /
// 6.8, 64 / 41, 364 / 254.
static int prerelax_fused(lbm_channel *h, double rhoepsl, int niter, bool hold, int *done, double *rhoerrmax)
{
    constexpr unsigned long long PENDING = ~0ull; // no fabs() has these bits
    constexpr unsigned long long UNKNOWN = 0x7ff8ull << 48; // a NaN
    int rc = LBM_OK;
    unsigned long long *stop = h->errbits + ERR_SLOTS * ERR_STRIDE;
    volatile unsigned long long *out = h->errout;
    for (int k = 0; k < niter; k++)
        out[k] = PENDING;
    int sent = 0, seen = 0;
    const int cur0 = h->cur;
    bool end = false;
    while (seen < niter && !end) {
        if (sent < niter && sent - seen < (hold && seen == 0 ? 1 : PRE_AHEAD)) {
            rc = launch_step(h, true, sent ? stop : nullptr);
            if (rc)
                break;
            sent++;
            hipLaunchKernelGGL(k_err_final, dim3(1), dim3(ERR_SLOTS), 0, h->stream, h->errbits, h->errout + sent - 1,
                               stop, rhoepsl, sent == 1);
            rc = dispatch_err(hipGetLastError(), "prerelax");
            if (rc) { // a step without its maximum
                out[sent - 1] = UNKNOWN;
                (void)hipMemsetAsync(h->errbits, 0, ERR_SLOTS * ERR_STRIDE * sizeof(unsigned long long), h->stream);
                break;
            }
            continue;
        }
        unsigned long long u;
        for (uint32_t spin = 1; (u = out[seen]) == PENDING; spin++) {
            if (spin % 1024)
                continue;
            const hipError_t e = hipStreamQuery(h->stream);
            if (e == hipErrorNotReady)
                continue;
            rc = dispatch_err(e, "prerelax");
            if (!rc && out[seen] == PENDING)
                rc = fail(LBM_ERR_HIP, "prerelax: no result of iteration %d", seen);
            if (rc)
                break;
        }
        if (rc)
            break;
        memcpy(&rhoerrmax[seen], &u, sizeof(u));
        end = rhoerrmax[seen] <= rhoepsl;
        seen++;
    }
    // what ran after the end had no effect; its results are written before the
    // next call's.  After an error the iterations in flight still take effect.
    if (sent > seen) {
        const hipError_t e = hipStreamSynchronize(h->stream);
        if (!rc)
            rc = dispatch_err(e, "prerelax");
        for (; !end && seen < sent && out[seen] != PENDING; seen++) {
            const unsigned long long u = out[seen];
            memcpy(&rhoerrmax[seen], &u, sizeof(u));
            end = rhoerrmax[seen] <= rhoepsl;
        }
    }
    h->cur = cur0 ^ (seen & 1);
    *done = seen;
    return rc;
}

int lbm_prerelax(lbm_channel *h, double rhoepsl, int niter, int *done, double *rhoerrmax)
{
    CHECK_H(h);
    if (niter < 1 || !done || !rhoerrmax)
        return fail(LBM_ERR_ARG, "lbm_prerelax: need niter >= 1, done and rhoerrmax");
    *done = 0;
    int rc = materialize(h);
    if (rc)
        return rc;
    const bool fused = !h->part && !h->mlp && !h->fc.tab && ensure_errout(h);
    while (*done < niter) {
        int n = 0;
        double *err = rhoerrmax + *done;
        if (fused) {
            rc = prerelax_fused(h, rhoepsl, std::min(niter - *done, PRE_ITERS), *done == 0, &n, err);
        } else {
            rc = lbm_rhoupdat(h, err);
            if (!rc)
                rc = launch_step(h);
            n = rc ? 0 : 1;
        }
        *done += n;
        if (rc)
            return rc;
        if (err[n - 1] <= rhoepsl)
            break;
    }
    return LBM_OK;
}

int lbm_avedensity(lbm_channel *h, double *rhomean)
{
    CHECK_H(h);
    double sum = 0.0, cnt = 0.0, mean;
    int rc;
    if (h->ms == FROM_CUR && h->rho_off == 0.0) {
        // rho is virtual: reduce macrovar(F) directly and keep the correction
        // as an offset applied by the next collision
        rc = reduce_rho(h, 1, &sum, &cnt);
        if (rc)
            return rc;
        mean = cnt > 0.0 ? sum / cnt : 0.0;
        h->rho_off = mean;
    } else {
        rc = materialize(h);
        if (rc)
            return rc;
        rc = reduce_rho(h, 0, &sum, &cnt);
        if (rc)
            return rc;
        mean = cnt > 0.0 ? sum / cnt : 0.0;
        hipLaunchKernelGGL(k_sub_scalar, dim3((unsigned)((h->g.N + 255) / 256)), dim3(256), 0, h->stream, h->mac[0],
                           h->g.N, mean);
        HIP_TRY(hipGetLastError());
    }
    h->fresh = false;
    if (rhomean)
        *rhomean = mean;
    return LBM_OK;
}

// Can the next two main-loop steps (collision_MRT + macrovar, twice) run as
// one blocked sweep?  Fused fields of the current lattice with no pending
// density offset, one uniform force, no particles, no closure.
static bool block_ready(const lbm_channel *h)
{
    return h->bK > 0 && !h->bskip && h->ms == FROM_CUR && h->rho_off == 0.0 && !h->part && !h->mlp &&
           h->fc.tab == nullptr && same_force(h->fm, h->fc);
}

// The force of one step of a pair: collision force fc, fields formed with fm
// (per node when the collision would run mode 16, as in launch_step).
static StepForce step_force_of(const lbm_channel *h, const ForceSpec &fc, const ForceSpec &fm)
{
    StepForce f;
    f.r = rates_of(h);
    f.r.fx = fc.fx;
    f.r.fy = fc.fy;
    f.r.fz = fc.fz;
    f.r = with_f32(f.r);
    f.fc = fc;
    f.fm = fm;
    f.per_node = (fc.tab != nullptr || !same_force(fm, fc)) ? 1 : 0;
    return f;
}

// Two main-loop steps in one blocked sweep (blocked.h): step t with force f0,
// step t+1 with f1; the handle's force (h->fc) is then step t+1's.
static int run_pair_with(lbm_channel *h, const StepForce &f0, const StepForce &f1)
{
    if (!h->bring) {
        const size_t rb = block_ring_elems(h->g, h->baxis, h->bK, h->bW, h->elem) * h->elem,
                     hb = block_head_elems(h->g, h->baxis, h->bW, h->elem) * h->elem;
        hipError_t e = hipMalloc(&h->bring, rb);
        if (e == hipSuccess)
            e = hipMalloc(&h->bhead, hb);
        if (e != hipSuccess) {
            if (h->bring)
                (void)hipFree(h->bring);
            h->bring = nullptr;
            return fail(LBM_ERR_NOMEM, "hipMalloc of the blocked-sweep ring (%zu + %zu bytes) failed: %s", rb, hb,
                        hipGetErrorString(e));
        }
    }
    const auto launches =
        block_schedule(h->g, h->baxis, f0, f1, h->bK, h->bW, h->lat[h->cur], h->lat[1 - h->cur], h->bring,
                       h->bhead, h->g.S, h->elem);
    for (const BlockArgs &a : launches) {
        int rc = dispatch_err(PREC_CALL(h, step_planes, a, h->baxis, h->stream), "collision (blocked sweep)");
        if (rc)
            return rc;
    }
    h->cur = 1 - h->cur;
    h->have_prev = false; // the other lattice holds the state two steps back
    h->fresh = false;
    fields_from_cur(h); // macrovar
    h->rho_off = 0.0;
    return LBM_OK;
}

// Two main-loop steps under the handle's uniform force.
static int run_pair(lbm_channel *h)
{
    const StepForce f = step_force_of(h, h->fc, h->fm);
    return run_pair_with(h, f, f);
}

// The force the main loop sets before the collision of step istep
// (Channel-Flow/main.f90:148-153 with the perturbation block switched on):
// FORCINGP while istep < npforcing, FORCING at istep == npforcing.
static int main_loop_force(lbm_channel *h, int istep, int npforcing, double force_in_y, double fy_forcing)
{
    if (istep < npforcing)
        return lbm_forcingp(h, istep, force_in_y);
    if (istep == npforcing)
        return lbm_set_force(h, 0.0, fy_forcing, 0.0);
    return LBM_OK;
}

int lbm_run_forcingp(lbm_channel *h, int istep0, int nsteps, int npforcing, double force_in_y, double fy_forcing)
{
    CHECK_H(h);
    if (nsteps < 0)
        return fail(LBM_ERR_ARG, "lbm_run_forcingp: nsteps %d < 0", nsteps);
    int s = 0;
    while (s < nsteps) {
        const int istep = istep0 + s + 1;
        int rc = main_loop_force(h, istep, npforcing, force_in_y, fy_forcing);
        if (rc)
            return rc;
        // a pair as one blocked sweep: fused fields of the current lattice,
        // no density offset, no particles or closure, and one uniform force
        // or, with bforced, any forces, evaluated per node
        bool paired = false;
        if (nsteps - s >= 2 && h->bK > 0 && !h->bskip && h->ms == FROM_CUR && h->rho_off == 0.0 && !h->part &&
            !h->mlp) {
            const ForceSpec fc0 = h->fc, fm0 = h->fm;
            rc = main_loop_force(h, istep + 1, npforcing, force_in_y, fy_forcing);
            if (rc)
                return rc;
            // step t+1's fields are macrovar of step t, formed with fc0
            const StepForce f0 = step_force_of(h, fc0, fm0), f1 = step_force_of(h, h->fc, fc0);
            if (h->bforced || (!f0.per_node && !f1.per_node)) {
                rc = run_pair_with(h, f0, f1);
                if (rc)
                    return rc;
                s += 2;
                paired = true;
            } else {
                h->fc = fc0; // step t alone; step t+1 sets its force again
                h->fm = fm0;
            }
        }
        if (!paired) {
            rc = launch_step(h);
            if (rc)
                return rc;
            fields_from_cur(h); // macrovar
            h->rho_off = 0.0;
            s += 1;
        }
    }
    return LBM_OK;
}

int lbm_run(lbm_channel *h, int nsteps)
{
    CHECK_H(h);
    if (nsteps < 0)
        return fail(LBM_ERR_ARG, "lbm_run: nsteps %d < 0", nsteps);
    int s = 0;
    while (nsteps - s >= 2 && block_ready(h)) {
        int rc = run_pair(h);
        if (rc)
            return rc;
        s += 2;
    }
    for (; s < nsteps; s++) {
        int rc = launch_step(h);
        if (rc)
            return rc;
        fields_from_cur(h); // macrovar
        h->rho_off = 0.0;
    }
    return LBM_OK;
}

int lbm_mass_sum(lbm_channel *h, double *mass)
{
    CHECK_H(h);
    if (!mass)
        return fail(LBM_ERR_ARG, "lbm_mass_sum: null output");
    SumArgs a;
    a.g = h->g;
    a.L = h->lat[h->cur];
    a.rho = nullptr;
    a.solid = solid_of(h);
    a.partials = h->partials;
    uint32_t grid = (uint32_t)std::min<uint64_t>(RED_BLOCKS, (h->g.N + 255) / 256);
    int rc = dispatch_err(PREC_CALL(h, mass_partials, a, grid, h->stream), "mass reduction");
    if (rc)
        return rc;
    rc = ensure_small(h);
    if (rc)
        return rc;
    hipLaunchKernelGGL(k_sum_ordered, dim3(1), dim3(256), 0, h->stream, (const double *)h->partials, grid,
                       results_at(h));
    HIP_TRY(hipGetLastError());
    rc = results(h, 1);
    if (rc)
        return rc;
    *mass = h->small[0];
    return LBM_OK;
}

int lbm_mass_sum_noalloc(lbm_channel *h, double *mass_dev)
{
    CHECK_H(h);
    if (!mass_dev)
        return fail(LBM_ERR_ARG, "lbm_mass_sum_noalloc: null output");
    // a kernel store through a host pointer would fault the GPU: accept only
    // device memory of this handle's GPU
    hipPointerAttribute_t at;
    if (hipPointerGetAttributes(&at, mass_dev) != hipSuccess || at.type != hipMemoryTypeDevice ||
        at.device != h->cfg.device) {
        (void)hipGetLastError();
        return fail(LBM_ERR_ARG, "lbm_mass_sum_noalloc: output %p is not device memory of device %d", (void *)mass_dev,
                    h->cfg.device);
    }
    double *part = g_scratch_ptr[h->cfg.device];
    if (!part)
        return fail(LBM_ERR_STATE, "lbm_mass_sum_noalloc: scratch of device %d not set up", h->cfg.device);
    SumArgs a;
    a.g = h->g;
    a.L = h->lat[h->cur];
    a.rho = nullptr;
    a.solid = solid_of(h);
    a.partials = part;
    // the same grid as lbm_mass_sum, so the two sums are equal bit for bit
    const uint32_t grid = (uint32_t)std::min<uint64_t>(RED_BLOCKS, (h->g.N + 255) / 256);
    if (grid > NOALLOC_PARTIALS) // cannot happen while RED_BLOCKS bounds the grid
        return fail(LBM_ERR_ARG, "lbm_mass_sum_noalloc: %u partials exceed the %u-double scratch", grid,
                    NOALLOC_PARTIALS);
    int rc = dispatch_err(PREC_CALL(h, mass_partials, a, grid, h->stream), "mass reduction");
    if (rc)
        return rc;
    hipLaunchKernelGGL(k_sum_ordered, dim3(1), dim3(256), 0, h->stream, (const double *)part, grid, mass_dev);
    HIP_TRY(hipGetLastError());
    return LBM_OK;
}

int lbm_statistc2(lbm_channel *h, double ustar, double ystar, double *out)
{
    CHECK_H(h);
    if (!out)
        return fail(LBM_ERR_ARG, "lbm_statistc2: null output");
    int rc = ensure_small(h);
    if (!rc)
        rc = plane_sums(h, results_at(h), false);
    if (!rc)
        rc = results(h, NPLANE * (size_t)h->g.lx);
    if (rc)
        return rc;
    stat_columns(h->g.lx, (double)h->g.ly * (double)h->g.lz, h->small, 1.0, ustar, ystar, out);
    return LBM_OK;
}

namespace {

// diag's block partials (q*grid + block) to totals in out[0..DIAG_Q).  The
// block brings the partials into LDS; the first thread of waves 0-6 adds a
// sum in increasing block order from 0.0, wave 7 merges the velocity maxima
// (larger value, then smaller node: any order gives the same) and waves 8, 9
// the density bounds.  One thread walking all of them in memory took 667 us; this takes 24 us.
__global__ void __launch_bounds__(64 * 10) k_diag_final(const double *__restrict__ part, uint32_t grid, double *out)
{
    __shared__ double p[DIAG_Q * DIAG_BLOCKS];
    for (uint32_t i = threadIdx.x; i < DIAG_Q * grid; i += blockDim.x)
        p[i] = part[i];
    __syncthreads();
    const uint32_t q = threadIdx.x >> 6, l = threadIdx.x & 63u;
    if (q < 7) {
        if (l != 0)
            return;
        double s = 0.0;
#pragma unroll 8
        for (uint32_t b = 0; b < grid; b++)
            s += p[q * grid + b];
        out[q] = s;
    } else if (q == 7) {
        double v = 0.0, vi = -1.0; // a block's own start: no node yet
        auto merge = [&](double ov, double oi) {
            if (ov > v || (ov == v && oi >= 0.0 && (vi < 0.0 || oi < vi))) {
                v = ov;
                vi = oi;
            }
        };
        for (uint32_t b = l; b < grid; b += 64)
            merge(p[7 * grid + b], p[8 * grid + b]);
        for (int o = 32; o > 0; o >>= 1) {
            const double ov = __shfl_xor(v, o), oi = __shfl_xor(vi, o);
            merge(ov, oi);
        }
        if (l == 0) {
            out[7] = v;
            out[8] = vi;
        }
    } else {
        const double *r = p + (q + 1) * grid; // 9: largest rho, 10: smallest
        double x = q == 8 ? -INFINITY : INFINITY;
        auto merge = [&](double o) { x = (q == 8 ? o > x : o < x) ? o : x; };
        for (uint32_t b = l; b < grid; b += 64)
            merge(r[b]);
        for (int o = 32; o > 0; o >>= 1)
            merge(__shfl_xor(x, o));
        if (l == 0)
            out[q + 1] = x;
    }
}

// vortcalc (Channel-Flow/saveload.f90:3929-4023) from the field arrays.
__global__ void k_vortcalc(Geom g, const double *__restrict__ ux, const double *__restrict__ uy,
                           const double *__restrict__ uz, const int *__restrict__ solid, const double *__restrict__ omg,
                           double *ox, double *oy, double *oz)
{
    const uint64_t n = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= g.N)
        return;
    if (solid && solid[n] >= 0) { // twice the particle's angular velocity
        const double *w = omg + 3 * (uint64_t)solid[n];
        ox[n] = 2.0 * w[0];
        oy[n] = 2.0 * w[1];
        oz[n] = 2.0 * w[2];
        return;
    }
    const uint64_t row = n / g.lx;
    const uint32_t i = (uint32_t)(n - row * g.lx);
    const uint32_t k = (uint32_t)(row / g.ly), j = (uint32_t)(row - (uint64_t)k * g.ly);
    const uint64_t plane = (uint64_t)g.lx * g.ly;
    double pwx, pvx;
    if (i == 0) { // wall forms of :3970-3975
        pwx = (3.0 * uz[n] + uz[n + 1]) / 3.0;
        pvx = (3.0 * uy[n] + uy[n + 1]) / 3.0;
    } else if (i == g.lx - 1) {
        pwx = -(3.0 * uz[n] + uz[n - 1]) / 3.0;
        pvx = -(3.0 * uy[n] + uy[n - 1]) / 3.0;
    } else {
        pwx = (uz[n + 1] - uz[n - 1]) / 2.0;
        pvx = (uy[n + 1] - uy[n - 1]) / 2.0;
    }
    // periodic images in y and z (exchng8, :4027-4054, on one rank)
    const uint64_t yp = j + 1 == g.ly ? n - (uint64_t)(g.ly - 1) * g.lx : n + g.lx;
    const uint64_t ym = j == 0 ? n + (uint64_t)(g.ly - 1) * g.lx : n - g.lx;
    const uint64_t zp = k + 1 == g.lz ? n - (uint64_t)(g.lz - 1) * plane : n + plane;
    const uint64_t zm = k == 0 ? n + (uint64_t)(g.lz - 1) * plane : n - plane;
    const double pwy = (uz[yp] - uz[ym]) / 2.0;
    const double puy = (ux[yp] - ux[ym]) / 2.0;
    const double puz = (ux[zp] - ux[zm]) / 2.0;
    const double pvz = (uy[zp] - uy[zm]) / 2.0;
    ox[n] = pwy - pvz;
    oy[n] = puz - pwx;
    oz[n] = pvx - puy;
}

} // namespace

int lbm_diag(lbm_channel *h, double ustar, double *out)
{
    CHECK_H(h);
    if (!out)
        return fail(LBM_ERR_ARG, "lbm_diag: null output");
    if (h->ms == FROM_PREV) {
        const int rc = materialize(h);
        if (rc)
            return rc;
    }
    DiagArgs a;
    a.g = h->g;
    a.L = h->lat[h->cur];
    a.rho = h->mac[0];
    a.ux = h->mac[1];
    a.uy = h->mac[2];
    a.uz = h->mac[3];
    a.solid = solid_of(h);
    a.f = h->fm;
    a.rho_off = h->rho_off;
    a.partials = h->partials;
    // DIAG_Q partials per block; the scratch holds at least 16 384 doubles
    const uint32_t grid = (uint32_t)std::min<uint64_t>(DIAG_BLOCKS, (h->g.N + 255) / 256);
    int rc = dispatch_err(PREC_CALL(h, diag_partials, a, h->ms == ARRAYS ? 0 : 1, grid, h->stream), "diag");
    if (rc)
        return rc;
    rc = ensure_small(h);
    if (rc)
        return rc;
    hipLaunchKernelGGL(k_diag_final, dim3(1), dim3(64 * 10), 0, h->stream, (const double *)h->partials, grid,
                       results_at(h));
    HIP_TRY(hipGetLastError());
    rc = results(h, DIAG_Q);
    if (rc)
        return rc;
    const double *t = h->small;
    // saveload.f90:1627-1640, in its order
    const double rn = t[6];
    double um = t[0] / rn, vm = t[1] / rn, wm = t[2] / rn;
    const double ur = sqrt(t[3] / rn - um * um), vr = sqrt(t[4] / rn - vm * vm), wr = sqrt(t[5] / rn - wm * wm);
    const long long idx = t[8] < 0.0 ? -1 : (long long)t[8];
    out[0] = t[7];
    out[1] = idx < 0 ? 0.0 : (double)(idx % h->g.lx + 1);
    out[2] = idx < 0 ? 0.0 : (double)((idx / h->g.lx) % h->g.ly + 1);
    out[3] = idx < 0 ? 0.0 : (double)(idx / ((long long)h->g.lx * h->g.ly) + 1);
    out[4] = um / ustar;
    out[5] = vm / ustar;
    out[6] = wm / ustar;
    out[7] = ur / ustar;
    out[8] = vr / ustar;
    out[9] = wr / ustar;
    out[10] = 1. - rn / ((double)h->g.lx * (double)h->g.ly * (double)h->g.lz);
    out[11] = t[9];
    out[12] = t[10];
    return LBM_OK;
}

int lbm_vortcalc(lbm_channel *h, double *ox, double *oy, double *oz)
{
    CHECK_H(h);
    if (!ox || !oy || !oz)
        return fail(LBM_ERR_ARG, "lbm_vortcalc: null output");
    int rc = materialize(h);
    if (rc)
        return rc;
    const size_t bytes = h->g.N * sizeof(double);
    double *d = nullptr;
    hipError_t e = hipMalloc((void **)&d, 3 * bytes);
    if (e != hipSuccess)
        return fail(LBM_ERR_NOMEM, "lbm_vortcalc: hipMalloc of %zu bytes failed: %s", 3 * bytes, hipGetErrorString(e));
    const double *omg = h->part ? h->part->ps.W : nullptr;
    hipLaunchKernelGGL(k_vortcalc, dim3((unsigned)((h->g.N + 255) / 256)), dim3(256), 0, h->stream, h->g,
                       (const double *)h->mac[1], (const double *)h->mac[2], (const double *)h->mac[3], solid_of(h),
                       omg, d, d + h->g.N, d + 2 * h->g.N);
    e = hipGetLastError();
    const HostPart parts[3] = {{ox, d, bytes}, {oy, d + h->g.N, bytes}, {oz, d + 2 * h->g.N, bytes}};
    if (e == hipSuccess)
        e = host_copy(h->cfg.device, h->stream, parts, 3, true);
    (void)hipFree(d);
    if (e != hipSuccess)
        return fail(LBM_ERR_HIP, "lbm_vortcalc: %s", hipGetErrorString(e));
    return LBM_OK;
}

int lbm_dissipation(lbm_channel *h, double tau, double ystar, double *out)
{
    CHECK_H(h);
    if (!out || !(tau > 0.0))
        return fail(LBM_ERR_ARG, "lbm_dissipation: need an output and tau > 0");
    if (h->ms == FROM_PREV) { // f is the current lattice's, the fields the previous macrovar's
        const int rc = materialize(h);
        if (rc)
            return rc;
    }
    const lbm_config &c = h->cfg;
    DissArgs a;
    a.g = h->g;
    a.L = h->lat[h->cur];
    a.rho = h->mac[0];
    a.ux = h->mac[1];
    a.uy = h->mac[2];
    a.uz = h->mac[3];
    a.solid = solid_of(h);
    a.f = h->fm;
    a.rho_off = h->rho_off;
    a.s1 = c.s1;
    a.s9 = c.s9;
    a.coef2 = c.coef2;
    a.coef3 = c.coef3;
    a.coef5 = c.coef5;
    a.ww1 = c.ww1;
    a.ww2 = c.ww2;
    a.c15tau = 1.5 / tau;
    a.partials = h->partials + 2 * RED_BLOCKS;
    const uint32_t rows = h->g.ly * h->g.lz;
    const uint32_t chunks = std::min<uint32_t>(PLANE_CHUNKS, rows);
    int rc = dispatch_err(PREC_CALL(h, dissipation_partials, a, h->ms == ARRAYS ? 0 : 1, chunks, h->stream),
                          "dissipation");
    if (rc)
        return rc;
    rc = ensure_small(h);
    if (rc)
        return rc;
    const uint32_t width = NDISS * h->g.lx;
    hipLaunchKernelGGL(k_sum_columns, dim3((width + SUM_COLS - 1) / SUM_COLS), dim3(SUM_COLS * SUM_ROWS), 0, h->stream,
                       a.partials, chunks, width, results_at(h), (double *)nullptr);
    HIP_TRY(hipGetLastError());
    rc = results(h, width);
    if (rc)
        return rc;
    const double *t = h->small;
    const int lx = h->g.lx;
    for (int i = 1; i <= lx; i++) { // saveload.f90:4857-4875
        const double nf = t[4 * (size_t)lx + i - 1];
        double yplus = ((double)i - 0.5) / ystar;
        if (i > lx / 2)
            yplus = ((double)(lx - i) + 0.5) / ystar;
        double *o = out + 6 * (size_t)(i - 1);
        o[0] = (double)i - 0.5;
        o[1] = yplus;
        for (int q = 0; q < 4; q++)
            o[2 + q] = t[(size_t)q * lx + i - 1] / nf;
    }
    return LBM_OK;
}

int lbm_stats_accumulate(lbm_channel *h)
{
    CHECK_H(h);
    int rc = plane_sums(h, h->red_out + 2, true);
    if (rc)
        return rc;
    h->stat_n++;
    return LBM_OK;
}

int lbm_stats_read(lbm_channel *h, double ustar, double ystar, double *out, long long *nsamples)
{
    CHECK_H(h);
    if (!out)
        return fail(LBM_ERR_ARG, "lbm_stats_read: null output");
    if (nsamples)
        *nsamples = h->stat_n;
    if (h->stat_n == 0)
        return fail(LBM_ERR_STATE, "lbm_stats_read: no samples accumulated");
    const int rc = read_small(h, h->stat_acc, NPLANE * (size_t)h->g.lx * sizeof(double));
    if (rc)
        return rc;
    stat_columns(h->g.lx, (double)h->g.ly * (double)h->g.lz, h->small, (double)h->stat_n, ustar, ystar, out);
    return LBM_OK;
}

int lbm_stats_accumulate_filtered(lbm_channel *h)
{
    CHECK_H(h);
    if (h->g.lx % 2 || h->g.ly % 2 || h->g.lz % 2)
        return fail(LBM_ERR_ARG, "lbm_stats_accumulate_filtered: the 2x2x2 filter needs even lx, ly, lz (%u, %u, %u)",
                    h->g.lx, h->g.ly, h->g.lz);
    if (h->part)
        return fail(LBM_ERR_STATE, "lbm_stats_accumulate_filtered: not defined with particles (filter cells would mix "
                                   "fluid and solid nodes)");
    if (!h->fstat_acc) {
        const uint64_t n = NPLANE * (uint64_t)(h->g.lx / 2);
        if (hipMalloc((void **)&h->fstat_acc, n * sizeof(double)) != hipSuccess)
            return fail(LBM_ERR_NOMEM, "hipMalloc of the filtered statistics accumulator failed");
        hipLaunchKernelGGL(k_fill, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, h->stream, h->fstat_acc, n, 0.0);
        HIP_TRY(hipGetLastError());
        h->fstat_n = 0;
    }
    int rc = filtered_plane_sums(h);
    if (rc)
        return rc;
    h->fstat_n++;
    return LBM_OK;
}

int lbm_stats_read_filtered(lbm_channel *h, double ustar, double ystar, double *out, long long *nsamples)
{
    CHECK_H(h);
    if (!out)
        return fail(LBM_ERR_ARG, "lbm_stats_read_filtered: null output");
    if (nsamples)
        *nsamples = h->fstat_n;
    if (h->fstat_n == 0)
        return fail(LBM_ERR_STATE, "lbm_stats_read_filtered: no samples accumulated");
    const uint32_t lxc = h->g.lx / 2;
    const int rc = read_small(h, h->fstat_acc, NPLANE * (size_t)lxc * sizeof(double));
    if (rc)
        return rc;
    stat_columns(lxc, (double)(h->g.ly / 2) * (double)(h->g.lz / 2), h->small, (double)h->fstat_n, ustar, ystar, out);
    return LBM_OK;
}

int lbm_stats_reset(lbm_channel *h)
{
    CHECK_H(h);
    const uint64_t n = NPLANE * (uint64_t)h->g.lx;
    hipLaunchKernelGGL(k_fill, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, h->stream, h->stat_acc, n, 0.0);
    HIP_TRY(hipGetLastError());
    h->stat_n = 0;
    if (h->fstat_acc) {
        const uint64_t nf = NPLANE * (uint64_t)(h->g.lx / 2);
        hipLaunchKernelGGL(k_fill, dim3((unsigned)((nf + 255) / 256)), dim3(256), 0, h->stream, h->fstat_acc, nf,
                           0.0);
        HIP_TRY(hipGetLastError());
    }
    h->fstat_n = 0;
    return LBM_OK;
}

int lbm_sync(lbm_channel *h)
{
    CHECK_H(h);
    HIP_TRY(hipStreamSynchronize(h->stream));
    return LBM_OK;
}

int lbm_time_steps(lbm_channel *h, int nsteps, double *avg_ms, double *total_ms)
{
    CHECK_H(h);
    if (nsteps <= 0)
        return fail(LBM_ERR_ARG, "lbm_time_steps: nsteps must be positive");
    // one timed unit per single step, or per blocked pair of steps; the
    // events are destroyed on every return path
    struct Events {
        std::vector<hipEvent_t> e;
        ~Events()
        {
            for (hipEvent_t x : e)
                if (x)
                    (void)hipEventDestroy(x);
        }
    } evs;
    evs.e.assign(2 * (size_t)nsteps, nullptr);
    std::vector<hipEvent_t> &ev = evs.e;
    for (auto &e : ev)
        HIP_TRY(hipEventCreate(&e));
    int rc = LBM_OK;
    int units = 0;
    for (int s = 0; s < nsteps && rc == LBM_OK; units++) {
        HIP_TRY(hipEventRecord(ev[2 * units], h->stream));
        if (nsteps - s >= 2 && block_ready(h)) {
            rc = run_pair(h);
            s += 2;
        } else {
            rc = launch_step(h);
            fields_from_cur(h);
            h->rho_off = 0.0;
            s += 1;
        }
        HIP_TRY(hipEventRecord(ev[2 * units + 1], h->stream));
    }
    if (rc == LBM_OK) {
        HIP_TRY(hipEventSynchronize(ev[2 * units - 1]));
        double sum = 0.0;
        for (int u = 0; u < units; u++) {
            float ms = 0.f;
            HIP_TRY(hipEventElapsedTime(&ms, ev[2 * u], ev[2 * u + 1]));
            sum += ms;
        }
        float tot = 0.f;
        HIP_TRY(hipEventElapsedTime(&tot, ev[0], ev[2 * units - 1]));
        if (avg_ms)
            *avg_ms = sum / nsteps; // device time per step
        if (total_ms)
            *total_ms = tot;
    }
    return rc;
}

int lbm_device_bytes(lbm_channel *h, size_t *bytes)
{
    if (!h || !bytes)
        return fail(LBM_ERR_ARG, "lbm_device_bytes: null argument");
    size_t b = 2 * (size_t)h->g.S * 19 * h->elem;
    if (h->mac[0])
        b += 4 * (size_t)h->g.N * sizeof(double);
    if (h->stage)
        b += STAGE_BYTES;
    if (h->bring)
        b += (block_ring_elems(h->g, h->baxis, h->bK, h->bW, h->elem) +
              block_head_elems(h->g, h->baxis, h->bW, h->elem)) * h->elem;
    b += (2 * RED_BLOCKS + (size_t)PLANE_CHUNKS * NPLANE * h->g.lx + 2 + 2 * NPLANE * (size_t)h->g.lx) * sizeof(double) + ERR_BYTES;
    *bytes = b;
    return LBM_OK;
}

int lbm_block_info(lbm_channel *h, int *axis, int *slabs)
{
    CHECK_H(h);
    if (axis)
        *axis = h->baxis == 2 ? 'z' : 'y';
    if (slabs)
        *slabs = (int)h->bK;
    return LBM_OK;
}

int lbm_block_pairs(lbm_channel *h, int *pairs)
{
    CHECK_H(h);
    if (!pairs)
        return fail(LBM_ERR_ARG, "lbm_block_pairs: null output");
    *pairs = h->bK > 0 && !h->bskip;
    return LBM_OK;
}

int lbm_block_rows(lbm_channel *h, int *rows)
{
    CHECK_H(h);
    if (!rows)
        return fail(LBM_ERR_ARG, "lbm_block_rows: null output");
    *rows = (int)h->bW;
    return LBM_OK;
}

// `count` stored values of population i at `v` as FP64.
static void widen(const lbm_channel *h, int i, const void *v, uint64_t count, double *o)
{
    if (h->prec == LBM_FP64) {
        memcpy(o, v, count * sizeof(double));
    } else if (h->prec == LBM_FP32) {
        const float *x = (const float *)v;
        for (uint64_t n = 0; n < count; n++)
            o[n] = x[n];
    } else if (h->prec == LBM_FP16) {
        const _Float16 *x = (const _Float16 *)v;
        const double sc = i == 0 ? 0.25 : (i <= 6 ? 1.0 / 16.0 : 1.0 / 32.0);
        for (uint64_t n = 0; n < count; n++)
            o[n] = (double)(float)x[n] * sc;
    } else {
        const uint16_t *x = (const uint16_t *)v;
        const float sc = FP16C_UP / fp16_scale_rt(i);
        for (uint64_t n = 0; n < count; n++)
            o[n] = (double)(fp16c_unpack(x[n]) * sc);
    }
}

// Nodes [n0, n0 + count) of the stored post-collision lattice as FP64,
// population-major (out[i*count + k] = P_i(n0 + k)), widened on the host.
static int download_post_range(lbm_channel *h, uint64_t n0, uint64_t count, double *out)
{
    const uint64_t S = h->g.S;
    const unsigned char *L = (const unsigned char *)h->lat[h->cur];
    const hipStream_t s = h->stream;
    HIP_TRY(hipStreamSynchronize(s));
    HostPool &pool = host_pool();
    std::unique_lock<std::mutex> lock(pool.mu, std::defer_lock);
    const int workers = host_workers(19 * count * sizeof(double), true);
    const bool sliced = 19 * count * h->elem >= HOST_MIN && !runtime_array(out);
    if (sliced && lock.try_lock() && pool.ready(h->cfg.device, workers)) {
        // populations start on lines, and each is read from the 16-byte word that
        // holds node n0 on: link_copy leaves other addresses to the runtime, 14 us
        // each (13 108 odd nodes in FP32: 301 us with 19 such copies)
        const uint64_t word = 16 / h->elem, lead = n0 % word, all = lead + count;
        const uint64_t per = HOST_SLICE / h->elem, m = (all + per - 1) / per; // slices of a population
        // one thread's short populations share a slot, up to five, for fewer waits
        const uint64_t row = (all + word - 1) / word * word;
        const uint64_t rows = workers > 1 ? 1 : std::max<uint64_t>(1, std::min<uint64_t>(5, per / row));
        const uint64_t nslices = rows > 1 ? (19 + rows - 1) / rows : 19 * m;
        const hipError_t e = host_slices_out(
            pool, h->cfg.device, s, nslices, workers,
            [&](size_t k, int, char *pinned, hipStream_t on) {
                hipError_t le = hipSuccess;
                const uint64_t at = k % m * per, i0 = k / m * rows;
                for (uint64_t i = i0; i < std::min<uint64_t>(19, i0 + rows) && le == hipSuccess; i++)
                    le = link_copy(pinned + (i - i0) * row * h->elem, L + (i * S + n0 - lead + at) * h->elem,
                                   std::min<uint64_t>(per, all - at) * h->elem, true, on);
                return le;
            },
            [&](size_t k, const char *pinned) {
                const uint64_t at = k % m * per, i0 = k / m * rows, skip = at == 0 ? lead : 0;
                for (uint64_t i = i0; i < std::min<uint64_t>(19, i0 + rows); i++)
                    widen(h, (int)i, pinned + ((i - i0) * row + skip) * h->elem,
                          std::min<uint64_t>(per, all - at) - skip, out + i * count + at + skip - lead);
            });
        if (e != hipSuccess)
            return fail(LBM_ERR_HIP, "lattice download: %s", hipGetErrorString(e));
        return LBM_OK;
    }
    if (h->prec == LBM_FP64) { // nothing to widen
        for (int i = 0; i < 19; i++)
            HIP_TRY(hipMemcpyAsync(out + (size_t)i * count, L + ((size_t)i * S + n0) * sizeof(double),
                                   count * sizeof(double), hipMemcpyDeviceToHost, s));
        HIP_TRY(hipStreamSynchronize(s));
        return LBM_OK;
    }
    std::vector<unsigned char> buf(count * h->elem);
    for (int i = 0; i < 19; i++) {
        HIP_TRY(hipMemcpyAsync(buf.data(), L + ((size_t)i * S + n0) * h->elem, count * h->elem,
                               hipMemcpyDeviceToHost, s));
        HIP_TRY(hipStreamSynchronize(s));
        widen(h, i, buf.data(), count, out + (size_t)i * count);
    }
    return LBM_OK;
}

int lbm_download_post(lbm_channel *h, double *post)
{
    CHECK_H(h);
    if (!post)
        return fail(LBM_ERR_ARG, "lbm_download_post: null output");
    return download_post_range(h, 0, h->g.N, post);
}

int lbm_download_post_range(lbm_channel *h, long long first, long long count, double *post)
{
    CHECK_H(h);
    if (!post)
        return fail(LBM_ERR_ARG, "lbm_download_post_range: null output");
    if (first < 0 || count < 0 || (unsigned long long)first + (unsigned long long)count > h->g.N)
        return fail(LBM_ERR_ARG, "lbm_download_post_range: nodes [%lld, %lld + %lld) outside the %llu-node lattice",
                    first, first, count, (unsigned long long)h->g.N);
    if (count == 0)
        return LBM_OK;
    return download_post_range(h, (uint64_t)first, (uint64_t)count, post);
}

static int part_alloc(Part *pt, void **p, size_t bytes)
{
    if (hipMalloc(p, bytes) != hipSuccess)
        return fail(LBM_ERR_NOMEM, "hipMalloc of particle state (%zu bytes) failed", bytes);
    pt->allocs.push_back(*p);
    return LBM_OK;
}

// The collision's flags after beads_links.
static int particles_inside(lbm_channel *h)
{
    const PartGeom &pg = h->part->pg;
    const PartState &ps = h->part->ps;
    const hipError_t e = h->prec == LBM_FP64   ? PartLaunch<0>::inside(pg, ps, h->stream)
                         : h->prec == LBM_FP32 ? PartLaunch<1>::inside(pg, ps, h->stream)
                         : h->prec == LBM_FP16 ? PartLaunch<2>::inside(pg, ps, h->stream)
                                               : PartLaunch<3>::inside(pg, ps, h->stream);
    return dispatch_err(e, "beads_links");
}

int lbm_particles_create(lbm_channel *h, const lbm_particle_config *pc, const double *pos, const double *vel,
                         const double *omg)
{
    CHECK_H(h);
    if (!pc || !pos)
        return fail(LBM_ERR_ARG, "lbm_particles_create: null argument");
    if (h->part)
        return fail(LBM_ERR_STATE, "lbm_particles_create: particles already exist on this handle");
    if (h->fc.tab)
        return fail(LBM_ERR_STATE, "lbm_particles_create: particles need a uniform force (FORCING, not FORCINGP)");
    if (pc->npart < 1 || !(pc->rad > 0.0) || !(pc->rhopart > 0.0) || pc->nave < 0)
        return fail(LBM_ERR_ARG, "lbm_particles_create: need npart >= 1, rad > 0, rhopart > 0, nave >= 0");
    if (!(pc->mingap > 0.0) || !(pc->mingap_w > 0.0) || !(pc->visc >= 0.0) ||
        (pc->visc > 0.0 && !(pc->lub_cut > pc->lub_min && pc->lub_min > 0.0)))
        return fail(LBM_ERR_ARG, "lbm_particles_create: need mingap, mingap_w > 0, visc >= 0 and, with visc > 0, "
                                 "lub_cut > lub_min > 0");
    const double lx = h->g.lx, ly = h->g.ly, lz = h->g.lz;
    for (int p = 0; p < pc->npart; p++) {
        const double *X = pos + 3 * p;
        if (!(X[0] - pc->rad > 0.0 && X[0] + pc->rad < lx) || !(X[1] >= 0.0 && X[1] < ly) ||
            !(X[2] >= 0.0 && X[2] < lz))
            return fail(LBM_ERR_ARG,
                        "lbm_particles_create: particle %d at (%g, %g, %g) must lie inside the channel "
                        "(R < x < lx - R, 0 <= y < ly, 0 <= z < lz)",
                        p, X[0], X[1], X[2]);
    }
    Part *pt = new Part();
    if ((PART_STATE * (size_t)pc->npart + 1) * sizeof(double) > small_bytes(h))
        pt->host.resize(PART_STATE * (size_t)pc->npart + 1);
    PartGeom &pg = pt->pg;
    PartState &ps = pt->ps;
    memset(&pg, 0, sizeof(pg));
    memset(&ps, 0, sizeof(ps));
    const double pi = 3.14159265358979323846;
    pg.g = h->g;
    pg.np = pc->npart;
    pg.R = pc->rad;
    pg.R2 = pc->rad * pc->rad;
    // cut links: about 5 per surface node; capacity with margin
    const double area = 4.0 * pi * (pc->rad + 1.0) * (pc->rad + 1.0);
    pg.maxlink = pc->maxlink > 0 ? pc->maxlink : (int)(12.0 * area) + 256;
    pg.maxfill = (int)(4.0 * area) + 64;
    pg.volume = 4.0 / 3.0 * pi * pc->rad * pc->rad * pc->rad;
    pg.mass = pc->rhopart * pg.volume;
    pg.inertia = 0.4 * pg.mass * pc->rad * pc->rad;
    pg.rhopart = pc->rhopart;
    pg.mingap = pc->mingap;
    pg.mingap_w = pc->mingap_w;
    pg.stf0 = pc->stf0;
    pg.stf1 = pc->stf1;
    pg.stf0_w = pc->stf0_w;
    pg.stf1_w = pc->stf1_w;
    pg.visc = pc->visc;
    pg.lub_cut = pc->lub_cut;
    pg.lub_min = pc->lub_min;
    pg.pressure_force = pc->pressure_force;
    pg.nave = pc->nave;
    pg.fx = h->fc.fx;
    pg.fy = h->fc.fy;
    pg.fz = h->fc.fz;
    const size_t np = pc->npart, nl = np * pg.maxlink, nf = np * pg.maxfill;
    int rc = LBM_OK;
    auto A = [&](void **p, size_t bytes) {
        if (rc == LBM_OK)
            rc = part_alloc(pt, p, bytes);
    };
    // what lbm_particles_get reads in one piece: X, the previous positions, V,
    // W, FH, TQ, FC, FL and the overflow word
    A((void **)&ps.X, (PART_STATE * np + 1) * sizeof(double));
    ps.V = ps.X + 6 * np;
    ps.W = ps.V + 3 * np;
    ps.FH = ps.W + 3 * np;
    ps.TQ = ps.FH + 3 * np;
    ps.FC = ps.TQ + 3 * np;
    ps.FL = ps.FC + 3 * np;
    ps.overflow = (int *)(ps.FL + 3 * np);
    A((void **)&ps.TH, 3 * np * sizeof(double));
    A((void **)&ps.Aprev, 3 * np * sizeof(double));
    A((void **)&ps.ALprev, 3 * np * sizeof(double));
    A((void **)&ps.FHprev, 3 * np * sizeof(double));
    A((void **)&ps.TQprev, 3 * np * sizeof(double));
    A((void **)&ps.VWnew, 6 * np * sizeof(double));
    A((void **)&ps.nsteps_done, sizeof(int));
    A((void **)&ps.solid, h->g.N * sizeof(int));
    const size_t inside_bytes = h->g.N * (h->elem == 2 ? sizeof(InsideFlag<2>) : sizeof(InsideFlag<0>));
    A((void **)&ps.inside, inside_bytes);
    A((void **)&ps.link_node, nl * sizeof(int));
    A((void **)&ps.link_dir, nl);
    A((void **)&ps.link_q, nl * sizeof(double));
    A((void **)&ps.link_contrib, nl * 6 * sizeof(double));
    A((void **)&ps.link_count, np * sizeof(int));
    A((void **)&ps.fill_node, nf * sizeof(int));
    A((void **)&ps.fill_count, np * sizeof(int));
    if (rc) {
        for (void *p : pt->allocs)
            (void)hipFree(p);
        delete pt;
        return rc;
    }
    std::vector<double> zero(3 * np, 0.0);
    HIP_TRY(hipMemcpyAsync(ps.X, pos, 3 * np * sizeof(double), hipMemcpyHostToDevice, h->stream));
    HIP_TRY(hipMemcpyAsync(ps.X + 3 * np, pos, 3 * np * sizeof(double), hipMemcpyHostToDevice, h->stream));
    HIP_TRY(hipMemcpyAsync(ps.V, vel ? vel : zero.data(), 3 * np * sizeof(double), hipMemcpyHostToDevice, h->stream));
    HIP_TRY(hipMemcpyAsync(ps.W, omg ? omg : zero.data(), 3 * np * sizeof(double), hipMemcpyHostToDevice, h->stream));
    for (double *d : {ps.TH, ps.Aprev, ps.ALprev, ps.FH, ps.TQ, ps.FC, ps.FL, ps.FHprev, ps.TQprev})
        HIP_TRY(hipMemcpyAsync(d, zero.data(), 3 * np * sizeof(double), hipMemcpyHostToDevice, h->stream));
    HIP_TRY(hipMemsetAsync(ps.nsteps_done, 0, sizeof(int), h->stream));
    HIP_TRY(hipMemsetAsync(ps.overflow, 0, sizeof(int), h->stream));
    HIP_TRY(hipMemsetAsync(ps.solid, 0xff, h->g.N * sizeof(int), h->stream)); // -1: fluid
    HIP_TRY(hipMemsetAsync(ps.inside, 0, inside_bytes, h->stream));
    HIP_TRY(hipMemsetAsync(ps.fill_count, 0, np * sizeof(int), h->stream));
    HIP_TRY(hipMemsetAsync(ps.link_count, 0, np * sizeof(int), h->stream));
    h->part = pt;
    h->ave_pending = false;
    rc = dispatch_err(part_classify(pg, ps, 1, h->stream), "beads_links");
    if (!rc)
        rc = particles_inside(h);
    if (rc)
        return rc;
    int ovf = 0;
    HIP_TRY(hipMemcpyAsync(&ovf, ps.overflow, sizeof(int), hipMemcpyDeviceToHost, h->stream));
    HIP_TRY(hipStreamSynchronize(h->stream));
    if (ovf)
        return fail(LBM_ERR_ARG, "lbm_particles_create: cut-link list overflow (maxlink %d)", pg.maxlink);
    return LBM_OK;
}

#define CHECK_P(h)                                                                       \
    do {                                                                                 \
        CHECK_H(h);                                                                      \
        if (!(h)->part)                                                                  \
            return fail(LBM_ERR_STATE, "%s: no particles on this handle", __func__);     \
    } while (0)

static int overflow_error(const lbm_channel *h, int ovf, const char *what)
{
    if (ovf & 2)
        return fail(LBM_ERR_STATE, "%s: a particle's position or velocity became non-finite (the run diverged)",
                    what);
    if (ovf)
        return fail(LBM_ERR_STATE, "%s: a per-particle link or refill list overflowed (maxlink %d, maxfill %d)",
                    what, h->part->pg.maxlink, h->part->pg.maxfill);
    return LBM_OK;
}

static int check_overflow(lbm_channel *h, const char *what)
{
    int rc = read_small(h, h->part->ps.overflow, sizeof(int)), ovf = 0;
    if (rc)
        return rc;
    memcpy(&ovf, h->small, sizeof(ovf));
    return overflow_error(h, ovf, what);
}

int lbm_beads_links(lbm_channel *h)
{
    CHECK_P(h);
    const int rc = dispatch_err(part_classify(h->part->pg, h->part->ps, 0, h->stream), "beads_links");
    return rc ? rc : particles_inside(h);
}

int lbm_beads_filling(lbm_channel *h)
{
    CHECK_P(h);
    Part *pt = h->part;
    hipError_t e = h->prec == LBM_FP64   ? PartLaunch<0>::refill(pt->pg, pt->ps, h->lat[h->cur], h->stream)
                   : h->prec == LBM_FP32 ? PartLaunch<1>::refill(pt->pg, pt->ps, h->lat[h->cur], h->stream)
                   : h->prec == LBM_FP16 ? PartLaunch<2>::refill(pt->pg, pt->ps, h->lat[h->cur], h->stream)
                                         : PartLaunch<3>::refill(pt->pg, pt->ps, h->lat[h->cur], h->stream);
    return dispatch_err(e, "beads_filling");
}

int lbm_beads_collision(lbm_channel *h)
{
    CHECK_P(h);
    Part *pt = h->part;
    hipError_t e = h->prec == LBM_FP64   ? PartLaunch<0>::ibb(pt->pg, pt->ps, h->lat[h->cur], false, h->stream)
                   : h->prec == LBM_FP32 ? PartLaunch<1>::ibb(pt->pg, pt->ps, h->lat[h->cur], false, h->stream)
                   : h->prec == LBM_FP16 ? PartLaunch<2>::ibb(pt->pg, pt->ps, h->lat[h->cur], false, h->stream)
                                         : PartLaunch<3>::ibb(pt->pg, pt->ps, h->lat[h->cur], false, h->stream);
    int rc = dispatch_err(e, "beads_collision");
    if (rc)
        return rc;
    return dispatch_err(part_sum(pt->pg, pt->ps, h->stream), "beads_collision sum");
}

int lbm_beads_move(lbm_channel *h)
{
    CHECK_P(h);
    Part *pt = h->part;
    pt->pg.fx = h->fc.fx;
    pt->pg.fy = h->fc.fy;
    pt->pg.fz = h->fc.fz;
    return dispatch_err(part_move(pt->pg, pt->ps, h->stream), "beads_move");
}

// Lattices above this size run the particle work beside the collision.
constexpr uint64_t PART_ASIDE_BYTES = 260000000ull;

int lbm_run_particles(lbm_channel *h, int istep0, int nsteps)
{
    CHECK_P(h);
    if (nsteps < 0)
        return fail(LBM_ERR_ARG, "lbm_run_particles: nsteps %d < 0", nsteps);
    // What follows from the bounce-back's link contributions alone (the force
    // sums, beads_move and beads_links) runs on a second stream beside the
    // collision, which reads no particle state but ps.inside; the refill, which
    // needs both, waits for them and brings ps.inside up to date.  So a step is
    // a chain of bounce-back, collision and refill.  The next bounce-back also
    // settles the refilled nodes.  Streams of the default priority.  us per
    // step, with the classification between the steps / beside the collision:
    // 250 spheres on 96x384x192, FP64 492 / 462, FP32 293 / 280; 2 000 on
    // 192x768x384, 3 715 / 3 655 and 2 150 / 2 075.
    // A short collision hides little and the streams' events cost 20 us, so
    // small lattices use one stream and larger blocks (two / one: 3 spheres on
    // 32x64x32, FP64 77 / 48, FP32 77 / 46; 20 on 64x100x90, 93 / 73 and 86 /
    // 60; 40 on 64x192x96, FP64 of 179 MB 112 / 102, FP32 of 90 MB 99 / 74; FP32
    // of 140 MB 116 / 95, of 239 MB 149 / 140; FP64 of 280 MB 152 / 156).
    const bool aside = h->pstreams ? h->pstreams == 2 : 19 * h->g.S * h->elem > PART_ASIDE_BYTES;
    if (aside && !h->pstream) {
        HIP_TRY(hipStreamCreateWithFlags(&h->pstream, hipStreamNonBlocking));
        for (hipEvent_t &e : h->pev)
            HIP_TRY(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    }
    Part *pt = h->part;
    const int nave = pt->pg.nave;
    // a step that the collision refuses moves nothing (later ones of the call
    // follow their own macrovar and are not refused)
    const int refused = nsteps > 0 ? step_check(h) : LBM_OK;
    if (refused)
        return refused;
    for (int s = 0; s < nsteps; s++) {
        // beads_collision: the bounce-back here, its sums below
        hipError_t e = h->prec == LBM_FP64   ? PartLaunch<0>::ibb(pt->pg, pt->ps, h->lat[h->cur], s > 0, h->stream)
                       : h->prec == LBM_FP32 ? PartLaunch<1>::ibb(pt->pg, pt->ps, h->lat[h->cur], s > 0, h->stream)
                       : h->prec == LBM_FP16 ? PartLaunch<2>::ibb(pt->pg, pt->ps, h->lat[h->cur], s > 0, h->stream)
                                             : PartLaunch<3>::ibb(pt->pg, pt->ps, h->lat[h->cur], s > 0, h->stream);
        int rc = dispatch_err(e, "beads_collision");
        if (rc)
            return rc;
        // avedensity after a step that is a multiple of nave (main.f90:163-167),
        // taken once this bounce-back has completed the fluid nodes'
        // populations; the collision below subtracts the mean
        if (h->ave_pending) {
            rc = lbm_avedensity(h, nullptr);
            if (rc)
                return rc;
            h->ave_pending = false;
        }
        // what the collision would make first reads state that the side stream moves
        if (h->ms == FROM_PREV) {
            rc = materialize(h);
            if (rc)
                return rc;
        }
        if (aside) {
            HIP_TRY(hipEventRecord(h->pev[0], h->stream));
            HIP_TRY(hipStreamWaitEvent(h->pstream, h->pev[0], 0));
        }
        pt->pg.fx = h->fc.fx; // beads_move's body force (pressure_force)
        pt->pg.fy = h->fc.fy;
        pt->pg.fz = h->fc.fz;
        rc = dispatch_err(part_advance(pt->pg, pt->ps, aside, aside ? h->pstream : h->stream), "beads_move and beads_links");
        // the join point; on every return below the main stream waits for it
        // first, so no later call races the side stream's writes
        if (aside)
            HIP_TRY(hipEventRecord(h->pev[1], h->pstream));
        if (!rc)
            rc = launch_step(h);
        if (rc) {
            if (aside)
                (void)hipStreamWaitEvent(h->stream, h->pev[1], 0);
            return rc;
        }
        fields_from_cur(h); // macrovar
        h->rho_off = 0.0;
        const long long istep = (long long)istep0 + s + 1;
        if (nave > 0 && istep % nave == 0)
            h->ave_pending = true;
        if (aside)
            HIP_TRY(hipStreamWaitEvent(h->stream, h->pev[1], 0));
        void *lat = h->lat[h->cur];
        e = h->prec == LBM_FP64   ? PartLaunch<0>::refill_inside(pt->pg, pt->ps, lat, h->stream)
            : h->prec == LBM_FP32 ? PartLaunch<1>::refill_inside(pt->pg, pt->ps, lat, h->stream)
            : h->prec == LBM_FP16 ? PartLaunch<2>::refill_inside(pt->pg, pt->ps, lat, h->stream)
                                  : PartLaunch<3>::refill_inside(pt->pg, pt->ps, lat, h->stream);
        rc = dispatch_err(e, "beads_filling");
        if (rc)
            return rc;
    }
    if (nsteps > 0) {
        const int rc = dispatch_err(part_finish(pt->pg, pt->ps, h->stream), "beads_filling");
        if (rc)
            return rc;
    }
    return check_overflow(h, "lbm_run_particles");
}

int lbm_particles_get(lbm_channel *h, double *pos, double *vel, double *omg, double *force, double *torque,
                      double *contact, double *lub)
{
    CHECK_P(h);
    // one copy (seven small ones and the check's took 127 us)
    const size_t n = 3 * (size_t)h->part->pg.np, bytes = (PART_STATE / 3 * n + 1) * sizeof(double);
    const double *all = nullptr;
    int rc;
    if (bytes <= small_bytes(h)) {
        rc = read_small(h, h->part->ps.X, bytes);
        all = h->small;
    } else {
        const HostPart part = {h->part->host.data(), h->part->ps.X, bytes};
        rc = copy_parts(h, &part, 1, true, "lbm_particles_get");
        all = h->part->host.data();
    }
    if (rc)
        return rc;
    double *dst[7] = {pos, vel, omg, force, torque, contact, lub};
    for (int k = 0; k < 7; k++)
        if (dst[k])
            memcpy(dst[k], all + (k == 0 ? 0 : k + 1) * n, n * sizeof(double));
    int ovf;
    memcpy(&ovf, all + PART_STATE / 3 * n, sizeof(ovf));
    return overflow_error(h, ovf, "lbm_particles_get");
}

int lbm_particles_links(lbm_channel *h, int *maxlink, int *counts, int *node, int *dir, double *q)
{
    CHECK_P(h);
    const PartGeom &pg = h->part->pg;
    const PartState &ps = h->part->ps;
    if (maxlink)
        *maxlink = pg.maxlink;
    const size_t nl = (size_t)pg.np * pg.maxlink;
    std::vector<signed char> d(dir ? nl : 0);
    const HostPart parts[4] = {{counts, ps.link_count, pg.np * sizeof(int)},
                               {node, ps.link_node, nl * sizeof(int)},
                               {q, ps.link_q, nl * sizeof(double)},
                               {dir ? d.data() : nullptr, ps.link_dir, nl}};
    const int rc = copy_parts(h, parts, 4, true, "lbm_particles_links");
    if (rc)
        return rc;
    for (size_t k = 0; k < d.size(); k++)
        dir[k] = d[k];
    return check_overflow(h, "lbm_particles_links");
}

int lbm_particles_solid(lbm_channel *h, int *solid)
{
    CHECK_P(h);
    if (!solid)
        return fail(LBM_ERR_ARG, "lbm_particles_solid: null output");
    const HostPart part = {solid, h->part->ps.solid, h->g.N * sizeof(int)};
    return copy_parts(h, &part, 1, true, "lbm_particles_solid");
}

int lbm_closure_set(lbm_channel *h, const float *params, double ystar)
{
    CHECK_H(h);
    if (!params || !(ystar > 0.0))
        return fail(LBM_ERR_ARG, "lbm_closure_set: need parameters and ystar > 0");
    if (h->prec == LBM_FP64)
        return fail(LBM_ERR_ARG, "lbm_closure_set: the closure runs in FP32 arithmetic (FP32/FP16 storage)");
    if (h->part)
        return fail(LBM_ERR_STATE, "lbm_closure_set: not combined with particles");
    if (!(params[MLP_NUTMIN] > -1.0f && params[MLP_NUTMIN] <= 0.0f))
        return fail(LBM_ERR_ARG, "lbm_closure_set: the nu_t/nu floor %g must lie in (-1, 0]",
                    (double)params[MLP_NUTMIN]);
    for (int j = 0; j < MLP_H; j++)
        if (!(fabsf(params[MLP_B1 + j]) <= MLP_BIAS_MAX && fabsf(params[MLP_B2 + j]) <= MLP_BIAS_MAX))
            return fail(LBM_ERR_ARG, "lbm_closure_set: hidden bias %d beyond +-%g (or not finite)", j,
                        (double)MLP_BIAS_MAX);
    // the parameters, then the constants and the FP16 weight image of the
    // fused evaluation (mlp.h, mlp_derive)
    std::vector<float> dev(MLP_DEV_TOTAL);
    std::copy(params, params + MLP_TOTAL, dev.begin());
    mlp_derive(params, dev.data());
    if (!h->mlp)
        HIP_TRY(hipMalloc((void **)&h->mlp, MLP_DEV_TOTAL * sizeof(float)));
    HIP_TRY(hipMemcpyAsync(h->mlp, dev.data(), MLP_DEV_TOTAL * sizeof(float), hipMemcpyHostToDevice, h->stream));
    HIP_TRY(hipStreamSynchronize(h->stream));
    h->mlp_inv_ystar = (float)(1.0 / ystar);
    h->mlp_yscale = params[MLP_SCALE + 9];
    return LBM_OK;
}

// Closure inputs (what 0) or nu_t/nu (what 1) of every node into host memory.
static int closure_eval(lbm_channel *h, float *out, int what, const char *name)
{
    CHECK_H(h);
    if (!out)
        return fail(LBM_ERR_ARG, "%s: null output", name);
    if (!h->mlp)
        return fail(LBM_ERR_STATE, "%s: no closure set (lbm_closure_set)", name);
    if (h->ms != FROM_CUR || h->rho_off != 0.0)
        return fail(LBM_ERR_STATE, "%s: the closure needs fields from macrovar (call lbm_macrovar first)", name);
    StepArgs a;
    memset(&a, 0, sizeof(a));
    a.g = h->g;
    a.src = h->lat[h->cur];
    a.r = rates_of(h);
    a.fc = h->fc;
    a.fm = h->fm;
    a.mlp = h->mlp;
    a.inv_ystar = h->mlp_inv_ystar;
    a.yscale = h->mlp_yscale;
    const size_t node_bytes = (what == 0 ? MLP_IN : 1) * sizeof(float);
    void *const arrays[1] = {out};
    // the inputs' stores are 40 bytes apart from lane to lane
    return nodes_to_host(h, arrays, 1, node_bytes, what == 0, name, [&](uint64_t n0, uint64_t cnt, char *dev, size_t, hipStream_t on) {
        return PREC_CALL(h, closure_eval, a, n0, cnt, (float *)dev, what, on);
    });
}

int lbm_closure_inputs(lbm_channel *h, float *feat) { return closure_eval(h, feat, 0, "lbm_closure_inputs"); }

int lbm_closure_nut(lbm_channel *h, float *nut) { return closure_eval(h, nut, 1, "lbm_closure_nut"); }

int lbm_closure_clear(lbm_channel *h)
{
    CHECK_H(h);
    if (h->mlp) {
        HIP_TRY(hipStreamSynchronize(h->stream));
        (void)hipFree(h->mlp);
        h->mlp = nullptr;
    }
    return LBM_OK;
}

#define CHECK_T(t)                                                   \
    do {                                                             \
        if (!(t))                                                    \
            return fail(LBM_ERR_ARG, "%s: null trainer", __func__);  \
        g_err[0] = 0;                                                \
        HIP_TRY(hipSetDevice((t)->device));                          \
    } while (0)

int lbm_trainer_create(int device, long long capacity, const float *params, lbm_trainer **out)
{
    g_err[0] = 0;
    if (!out || !params || capacity < 1 || capacity > (1ll << 31))
        return fail(LBM_ERR_ARG, "lbm_trainer_create: need params, out and 1 <= capacity <= 2^31");
    *out = nullptr;
    HIP_TRY(hipSetDevice(device));
    lbm_trainer *t = new lbm_trainer();
    memset(t, 0, sizeof(*t));
    host_pool().retain();
    t->device = device;
    t->capacity = capacity;
    t->max_waves = 1u << 16;
    auto cleanup = [&](int code) {
        lbm_trainer_destroy(t);
        return code;
    };
    if (hipStreamCreateWithFlags(&t->stream, hipStreamNonBlocking) != hipSuccess)
        return cleanup(fail(LBM_ERR_HIP, "lbm_trainer_create: stream creation failed"));
    if (hipMalloc((void **)&t->feat, (size_t)capacity * MLP_IN * sizeof(float)) != hipSuccess ||
        hipMalloc((void **)&t->target, (size_t)capacity * sizeof(float)) != hipSuccess ||
        hipMalloc((void **)&t->w, MLP_TOTAL * sizeof(float)) != hipSuccess ||
        hipMalloc((void **)&t->m, MLP_NPARAM * sizeof(float)) != hipSuccess ||
        hipMalloc((void **)&t->v, MLP_NPARAM * sizeof(float)) != hipSuccess ||
        hipMalloc((void **)&t->partial, (size_t)MLP_GRAD_BLOCKS * (MLP_NPARAM + 1) * sizeof(float)) != hipSuccess ||
        hipMalloc((void **)&t->grad, (MLP_NPARAM + 1) * sizeof(float)) != hipSuccess)
        return cleanup(fail(LBM_ERR_NOMEM, "lbm_trainer_create: device allocation failed"));
    t->small = (float *)small_alloc(MLP_TOTAL * sizeof(float), &t->small_pinned);
    if (!t->small)
        return cleanup(fail(LBM_ERR_NOMEM, "lbm_trainer_create: allocation of the result buffer failed"));
    if (hipMemcpyAsync(t->w, params, MLP_TOTAL * sizeof(float), hipMemcpyHostToDevice, t->stream) != hipSuccess ||
        hipMemsetAsync(t->m, 0, MLP_NPARAM * sizeof(float), t->stream) != hipSuccess ||
        hipMemsetAsync(t->v, 0, MLP_NPARAM * sizeof(float), t->stream) != hipSuccess ||
        hipStreamSynchronize(t->stream) != hipSuccess)
        return cleanup(fail(LBM_ERR_HIP, "lbm_trainer_create: initialisation failed"));
    *out = t;
    return LBM_OK;
}

int lbm_trainer_destroy(lbm_trainer *t)
{
    if (!t)
        return LBM_OK;
    (void)hipSetDevice(t->device);
    if (t->stream)
        (void)hipStreamSynchronize(t->stream);
    for (void *p : {(void *)t->feat, (void *)t->target, (void *)t->w, (void *)t->m, (void *)t->v, (void *)t->partial,
                    (void *)t->grad})
        if (p)
            (void)hipFree(p);
    small_free(t->small, t->small_pinned);
    host_pool().release(); // before the trainer's own stream goes
    if (t->stream)
        (void)hipStreamDestroy(t->stream);
    delete t;
    return LBM_OK;
}

int lbm_trainer_add_filtered(lbm_trainer *t, lbm_channel *fine, double nu_coarse, double s9_coarse,
                             double ystar_coarse, long long *added)
{
    CHECK_T(t);
    if (!fine)
        return fail(LBM_ERR_ARG, "lbm_trainer_add_filtered: null channel");
    {
        HIP_TRY(hipSetDevice(fine->cfg.device));
        const int frc = flush_pending(fine);
        if (frc)
            return frc;
    }
    if (fine->cfg.device != t->device)
        return fail(LBM_ERR_ARG, "lbm_trainer_add_filtered: channel and trainer on different devices");
    if ((fine->g.lx | fine->g.ly | fine->g.lz) & 1)
        return fail(LBM_ERR_ARG, "lbm_trainer_add_filtered: fine grid %u x %u x %u must be even", fine->g.lx,
                    fine->g.ly, fine->g.lz);
    if (fine->part)
        return fail(LBM_ERR_ARG, "lbm_trainer_add_filtered: not for particle-laden channels");
    if (fine->fc.tab)
        return fail(LBM_ERR_ARG, "lbm_trainer_add_filtered: the fine channel needs a uniform force (FORCING)");
    const uint32_t lxc = fine->g.lx / 2, lyc = fine->g.ly / 2, lzc = fine->g.lz / 2;
    const long long Nc = (long long)lxc * lyc * lzc;
    if (t->count + Nc > t->capacity)
        return fail(LBM_ERR_ARG, "lbm_trainer_add_filtered: %lld samples would exceed the capacity %lld",
                    t->count + Nc, t->capacity);
    HIP_TRY(hipStreamSynchronize(fine->stream));
    // 10 filtered fields, then (per-plane targets) tau:S and S:S per node
    const bool plane = (t->target_mode == LBM_TARGET_PLANE);
    float *fields = nullptr;
    HIP_TRY(hipMalloc((void **)&fields, (size_t)Nc * (plane ? 12 : 10) * sizeof(float)));
    FilterArgs fa;
    fa.gf = fine->g;
    fa.L = fine->lat[fine->cur];
    fa.fx = fine->fc.fx;
    fa.fy = fine->fc.fy;
    fa.fz = fine->fc.fz;
    fa.lxc = lxc;
    fa.lyc = lyc;
    fa.lzc = lzc;
    fa.out = fields;
    hipError_t e = fine->prec == LBM_FP64   ? MlpLaunch<0>::filter(fa, t->stream)
                   : fine->prec == LBM_FP32 ? MlpLaunch<1>::filter(fa, t->stream)
                   : fine->prec == LBM_FP16 ? MlpLaunch<2>::filter(fa, t->stream)
                                            : MlpLaunch<3>::filter(fa, t->stream);
    FeatArgs ft;
    ft.lx = lxc;
    ft.ly = lyc;
    ft.lz = lzc;
    ft.fields = fields;
    ft.nu = (float)nu_coarse;
    ft.s9 = (float)s9_coarse;
    ft.inv_ystar = (float)(1.0 / ystar_coarse);
    std::vector<float> hp(MLP_TOTAL);
    if (e == hipSuccess)
        e = hipMemcpyAsync(hp.data(), t->w, MLP_TOTAL * sizeof(float), hipMemcpyDeviceToHost, t->stream);
    if (e == hipSuccess)
        e = hipStreamSynchronize(t->stream);
    ft.yscale = hp[MLP_SCALE + 9];
    ft.scale = t->w + MLP_SCALE;
    ft.feat = t->feat;
    ft.target = t->target;
    ft.offset = (uint64_t)t->count;
    ft.ts = plane ? fields + (size_t)Nc * 10 : nullptr;
    ft.ss = plane ? fields + (size_t)Nc * 11 : nullptr;
    if (e == hipSuccess)
        e = mlp_features(ft, t->stream);
    if (e == hipSuccess && plane)
        e = mlp_plane_targets(lxc, lyc, lzc, ft.ts, ft.ss, ft.nu, t->target, ft.offset, t->stream);
    if (e == hipSuccess)
        e = hipStreamSynchronize(t->stream);
    (void)hipFree(fields);
    if (e != hipSuccess)
        return fail(LBM_ERR_HIP, "lbm_trainer_add_filtered: %s", hipGetErrorString(e));
    t->count += Nc;
    if (added)
        *added = Nc;
    return LBM_OK;
}

int lbm_trainer_set_target(lbm_trainer *t, int mode)
{
    CHECK_T(t);
    if (mode != LBM_TARGET_LOCAL && mode != LBM_TARGET_PLANE)
        return fail(LBM_ERR_ARG, "lbm_trainer_set_target: mode %d is neither LBM_TARGET_LOCAL nor LBM_TARGET_PLANE",
                    mode);
    t->target_mode = mode;
    return LBM_OK;
}

int lbm_trainer_set_plane_targets(lbm_trainer *t, long long first, long long count, int nx, const float *values)
{
    CHECK_T(t);
    if (!values || nx < 1 || first < 0 || count < 0 || first + count > t->count)
        return fail(LBM_ERR_ARG, "lbm_trainer_set_plane_targets: need values, nx >= 1 and samples within the %lld held",
                    t->count);
    for (int i = 0; i < nx; i++)
        if (!std::isfinite(values[i]))
            return fail(LBM_ERR_ARG, "lbm_trainer_set_plane_targets: value %d is not finite", i);
    if (count == 0)
        return LBM_OK;
    float *dv = nullptr;
    HIP_TRY(hipMalloc((void **)&dv, (size_t)nx * sizeof(float)));
    hipError_t e = hipMemcpyAsync(dv, values, (size_t)nx * sizeof(float), hipMemcpyHostToDevice, t->stream);
    if (e == hipSuccess)
        e = mlp_fill_plane_targets(t->target, (uint64_t)first, (uint64_t)count, (uint32_t)nx, dv, t->stream);
    if (e == hipSuccess)
        e = hipStreamSynchronize(t->stream);
    (void)hipFree(dv);
    if (e != hipSuccess)
        return fail(LBM_ERR_HIP, "lbm_trainer_set_plane_targets: %s", hipGetErrorString(e));
    return LBM_OK;
}

// Most threads of a trainer's downloads, which are few: fewer slots to allocate,
// and no second stream (600 000 samples added, read back and destroyed: 4 330 us
// with six threads and two streams, 2 970-3 170 with these, 3 290 by the runtime).
static constexpr int TRAINER_COPY_THREADS = 4;

int lbm_trainer_add_samples(lbm_trainer *t, const float *features, const float *targets, long long n)
{
    CHECK_T(t);
    if (!features || !targets || n < 0 || t->count + n > t->capacity)
        return fail(LBM_ERR_ARG, "lbm_trainer_add_samples: bad arguments or capacity exceeded");
    // by the runtime: a trainer is filled in few calls, and the slots take longer
    // to allocate and give back than they save (900 000 samples, from creation to
    // destruction: 7 100 us with them, 2 040 without)
    HIP_TRY(hipMemcpyAsync(t->feat + (size_t)t->count * MLP_IN, features, (size_t)n * MLP_IN * sizeof(float),
                           hipMemcpyHostToDevice, t->stream));
    HIP_TRY(hipMemcpyAsync(t->target + t->count, targets, (size_t)n * sizeof(float), hipMemcpyHostToDevice,
                           t->stream));
    HIP_TRY(hipStreamSynchronize(t->stream));
    t->count += n;
    return LBM_OK;
}

int lbm_trainer_samples(lbm_trainer *t, long long *n, float *features, float *targets)
{
    CHECK_T(t);
    if (n)
        *n = t->count;
    const HostPart parts[2] = {{features, t->feat, (size_t)t->count * MLP_IN * sizeof(float)},
                               {targets, t->target, (size_t)t->count * sizeof(float)}};
    HIP_TRY(host_copy(t->device, t->stream, parts, 2, true, TRAINER_COPY_THREADS));
    return LBM_OK;
}

static int trainer_range(lbm_trainer *t, long long first, long long count, const char *fn)
{
    if (first < 0 || count < 1 || first + count > t->count)
        return fail(LBM_ERR_ARG, "%s: samples [%lld, %lld) outside [0, %lld)", fn, first, first + count, t->count);
    return LBM_OK;
}

// One gradient pass covers at most max_waves times 64 samples.
static int trainer_batch(lbm_trainer *t, long long batch, const char *fn)
{
    if ((batch + 63) / 64 > (long long)t->max_waves)
        return fail(LBM_ERR_ARG, "%s: batch of %lld samples exceeds %u waves of 64", fn, batch, t->max_waves);
    return LBM_OK;
}

int lbm_trainer_grad(lbm_trainer *t, long long first, long long count, float *grad, float *loss)
{
    CHECK_T(t);
    int rc = trainer_range(t, first, count, "lbm_trainer_grad");
    if (!rc)
        rc = trainer_batch(t, count, "lbm_trainer_grad");
    if (rc)
        return rc;
    HIP_TRY(mlp_grad(t->w, t->feat, t->target, (uint32_t)first, (uint32_t)count, t->partial, t->grad, t->w, t->m,
                     t->v, 1, 0.0f, 0, t->stream));
    HIP_TRY(small_copy(t->small, t->small_pinned, t->grad, (MLP_NPARAM + 1) * sizeof(float), t->stream));
    if (grad)
        memcpy(grad, t->small, MLP_NPARAM * sizeof(float));
    if (loss)
        *loss = t->small[MLP_NPARAM];
    return LBM_OK;
}

int lbm_trainer_train(lbm_trainer *t, long long first, long long count, int iterations, long long batch, float lr,
                      float *loss)
{
    CHECK_T(t);
    int rc = trainer_range(t, first, count, "lbm_trainer_train");
    if (rc)
        return rc;
    if (iterations < 1 || batch < 1 || batch > count)
        return fail(LBM_ERR_ARG, "lbm_trainer_train: need iterations >= 1 and 1 <= batch <= count");
    rc = trainer_batch(t, batch, "lbm_trainer_train");
    if (rc)
        return rc;
    long long pos = 0;
    for (int it = 0; it < iterations; it++) {
        if (pos + batch > count)
            pos = 0;
        t->step++;
        HIP_TRY(mlp_grad(t->w, t->feat, t->target, (uint32_t)(first + pos), (uint32_t)batch, t->partial, t->grad,
                         t->w, t->m, t->v, t->step, lr, 1, t->stream));
        pos += batch;
    }
    HIP_TRY(small_copy(t->small, t->small_pinned, t->grad + MLP_NPARAM, sizeof(float), t->stream));
    if (loss)
        *loss = t->small[0];
    return LBM_OK;
}

int lbm_trainer_predict(lbm_trainer *t, long long first, long long count, float *out)
{
    CHECK_T(t);
    if (!out || first < 0 || count < 1 || first + count > t->count)
        return fail(LBM_ERR_ARG, "lbm_trainer_predict: bad range or null output");
    // as nodes_to_host: the kernel stores into the pinned slots
    const size_t total = (size_t)count * sizeof(float);
    const int workers = std::min(TRAINER_COPY_THREADS, host_workers(total, true));
    const bool sliced = total >= HOST_MIN && !runtime_array(out);
    hipError_t e = sliced ? hipStreamSynchronize(t->stream) : hipSuccess;
    HostPool &pool = host_pool();
    std::unique_lock<std::mutex> lock(pool.mu, std::defer_lock);
    if (e == hipSuccess && sliced && lock.try_lock() && pool.ready(t->device, workers)) {
        const size_t per = host_slice(total, true) / sizeof(float), n = ((size_t)count + per - 1) / per;
        auto here = [&](size_t k) { return std::min<size_t>(per, (size_t)count - k * per); };
        e = host_slices_out(
            pool, t->device, t->stream, n, workers,
            [&](size_t k, int, char *pinned, hipStream_t on) {
                return mlp_predict(t->w, t->feat, (uint32_t)(first + k * per), (uint32_t)here(k), (float *)pinned, on);
            },
            [&](size_t k, const char *pinned) { memcpy(out + k * per, pinned, here(k) * sizeof(float)); });
    } else if (e == hipSuccess) {
        float *d = nullptr;
        e = hipMalloc((void **)&d, total);
        if (e == hipSuccess)
            e = mlp_predict(t->w, t->feat, (uint32_t)first, (uint32_t)count, d, t->stream);
        if (e == hipSuccess)
            e = hipMemcpyAsync(out, d, total, hipMemcpyDeviceToHost, t->stream);
        if (e == hipSuccess)
            e = hipStreamSynchronize(t->stream);
        (void)hipFree(d);
    }
    if (e != hipSuccess)
        return fail(LBM_ERR_HIP, "lbm_trainer_predict: %s", hipGetErrorString(e));
    return LBM_OK;
}

int lbm_trainer_params(lbm_trainer *t, float *params)
{
    CHECK_T(t);
    if (!params)
        return fail(LBM_ERR_ARG, "lbm_trainer_params: null output");
    HIP_TRY(small_copy(t->small, t->small_pinned, t->w, MLP_TOTAL * sizeof(float), t->stream));
    memcpy(params, t->small, MLP_TOTAL * sizeof(float));
    return LBM_OK;
}

} // extern "C"
