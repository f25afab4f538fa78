// batch.hip -- many independent DIAG- or MIXED-form problems of uneven size (nx, ny,
// N, ne, lambda, faces) solved together.
//
// Every problem is the five-stage pipeline of a solve:
//   0 R2C along y (+ faces)   1 C2C along x (+ faces)   2 mode solve (diagonalised, or MIXED)
//   3 C2C^-1 along x          4 C2R along y
// split into tasks: a tile of spectral columns of the mode solve, or one
// uniform-base tile of a transform pass (the standalone transform kernels'
// tiles; 256 copies for a length-1 pass).
//
// Staged variant: one launch per stage and task kind (the launch boundary
// is the dependency), recorded in a HIP graph that later solves replay.
// Fused variant (built, switched off -- see kVariants): ONE cooperative
// launch for the whole batch.  The stages run
// in order, separated by the runtime's grid barrier; the tasks of a stage,
// all kinds together, are dealt from per-XCD ranges by atomic counters.  The
// launch API checks that every work-group is resident, and every work-group
// runs the same stage loop, so each barrier is reached by all of them.
//
// One-element Dirichlet problems in DIAG form leave this scheme where the
// z-first kernels (zfirst.hip) hold them: three stages of lists, launched ahead
// of the rest in every variant.
//
// The autotuner times the usable variants (staged or fused, mode-solve tile
// height 32 or 64 rows) on the first solve of a batch shape and keeps the
// fastest.
#include "diag_waves_body.h"
#include "fft_body.h"
#include "mixed_body.h"

#include <hip/hip_cooperative_groups.h>

#include <array>
#include <map>
#include <mutex>
#include <string>
#include <vector>

namespace hz {

constexpr int kStages = 5;

struct BatchProblem {
    FftArgs f[4];    // passes 0..3 of xy_pass_args
    DiagArgs d;      // DIAG plans
    MixedArgs m;     // MIXED plans
    int ly, lx;      // transform lengths along y, x
    // 2 * (NP / 32 - 1) + general (NP = 32, 64, 96, 128), + 8 for a MIXED plan;
    // 16, 17 (N - 2 to 16, to 32) for what diag_waves.hip solves, 18 for a MIXED
    // plan of mixed_by_four_waves
    int dkind;
};

namespace {

// ---- fused variant: one cooperative launch ------------------------------------
// A transform task: uniform-base tile t of a pass of length L (W lanes per
// tile, as the staged launches use), or 256 copies of a length-1 pass.  A
// tile past the problem's table (a face tile of a problem without faces)
// does nothing.
template <int KIND>
__device__ __noinline__ void coop_fft(const FftArgs &a, int L, int t, double *smem)
{
    if (L == 1) {
        unit_line_element<KIND>(a, (long long)t * 256 + threadIdx.x);
        return;
    }
    const int W = L <= 16 ? 64 : L <= 64 ? 32 : 16;
    const long long tiles = uniform_main_tiles(a.nbatch, a.lanes, a.in_batch_stride, a.out_batch_stride, W) +
                            (long long)a.xlanes * ((a.nbatch + W - 1) / W);
    if (t >= tiles) return;
    switch (L) {
    case 16: fft_tile_uniform<16, 4, 4, 64, KIND>(a, t, smem); break;
    case 32: fft_tile_uniform<32, 8, 4, 32, KIND>(a, t, smem); break;
    case 64: fft_tile_uniform<64, 8, 8, 32, KIND>(a, t, smem); break;
    case 128: fft_tile_uniform<128, 16, 8, 16, KIND>(a, t, smem); break;
    default: fft_tile_uniform<256, 16, 16, 16, KIND>(a, t, smem); break;
    }
}

template <int NJ, int RT, bool GENERAL>
__device__ __forceinline__ void coop_diag_t(const DiagArgs &a, int t, double *smem)
{
    diag_tile<NJ, RT, GENERAL, false>(a, t, *reinterpret_cast<DiagShared<NJ, RT, GENERAL, false> *>(smem));
}

// A mode-solve task: tile t of the problem's DIAG kernel body (kinds 0, 2-7; a
// batch with other kinds is not run fused, see variant_usable).
template <int RT>
__device__ __noinline__ void coop_modes(const BatchProblem &pr, int t, double *smem)
{
    switch (pr.dkind) {
    case 0: coop_diag_t<2, RT, false>(pr.d, t, smem); break;
    case 2: coop_diag_t<4, RT, false>(pr.d, t, smem); break;
    case 3: coop_diag_t<4, RT, true>(pr.d, t, smem); break;
    case 4: coop_diag_t<6, RT, false>(pr.d, t, smem); break;
    case 5: coop_diag_t<6, RT, true>(pr.d, t, smem); break;
    case 6: coop_diag_t<8, RT, false>(pr.d, t, smem); break;
    default: coop_diag_t<8, RT, true>(pr.d, t, smem); break;
    }
}

template <int RT>
__device__ __forceinline__ void coop_task(const BatchProblem &pr, int s, int t, double *smem)
{
    switch (s) {
    case 0: coop_fft<FFT_R2C>(pr.f[0], pr.ly, t, smem); break;
    case 1: coop_fft<FFT_C2C_FWD>(pr.f[1], pr.lx, t, smem); break;
    case 2: coop_modes<RT>(pr, t, smem); break;
    case 3: coop_fft<FFT_C2C_INV>(pr.f[2], pr.lx, t, smem); break;
    default: coop_fft<FFT_C2R>(pr.f[3], pr.ly, t, smem); break;
    }
}

template <class T>
constexpr size_t cmax(T a, T b) { return a > b ? a : b; }

// Dynamic LDS of the fused kernel: the largest task body it may run.
template <int RT>
constexpr size_t coop_lds()
{
    size_t m = sizeof(double) * (256 + 2) * 16;  // transform tile, L = 256, W = 16
    m = cmax(m, sizeof(double) * (64 + 2) * 32);
    m = cmax(m, sizeof(double) * (16 + 2) * 64);
    m = cmax(m, sizeof(DiagShared<2, RT, false, false>));
    m = cmax(m, sizeof(DiagShared<4, RT, true, false>));
    m = cmax(m, sizeof(DiagShared<6, RT, true, false>));
    m = cmax(m, sizeof(DiagShared<8, RT, true, false>));
    return m;
}

// One persistent launch of the whole batch, launched cooperatively (every
// work-group resident, which the runtime checks at launch).  The stages run
// in order with a grid barrier between them; within a stage the tasks are
// independent.  xoff[s*(kXcds+1) + x] .. [.. + x + 1] is XCD x's contiguous
// range of the stage's task list (a share of every task kind); a work-group
// takes tasks from its own XCD's range through that range's counter
// ctr[s*kXcds + x], then helps drain the other XCDs' ranges.  The counters
// start at zero: each stage's are cleared after the barrier that ends it
// (the last stage's at the start of the next launch, four barriers before
// they are used).  Every work-group runs the same stage loop, so each reaches
// every barrier.  ctl[1] is set if the launch was not cooperative (no work
// is done then).
template <int RT>
__global__ __launch_bounds__(256, 2) void batch_coop_kernel(const BatchProblem *__restrict__ P,
                                                            const int2 *__restrict__ list,
                                                            const int *__restrict__ xoff, int *ctr, int *ctl)
{
    extern __shared__ double smem[];
    __shared__ int s_task;
    if (!cooperative_groups::this_grid().is_valid()) {
        if (blockIdx.x == 0 && threadIdx.x == 0) atomicOr(&ctl[1], 1);
        return;
    }
    const int home = blockIdx.x % kXcds;  // work-groups are dealt round-robin to the XCDs
    if (blockIdx.x == 0 && threadIdx.x < kXcds)
        __hip_atomic_store(&ctr[(kStages - 1) * kXcds + threadIdx.x], 0, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
    for (int s = 0; s < kStages; ++s) {
        const int *xo = xoff + s * (kXcds + 1);
        for (int k = 0; k < kXcds; ++k) {
            const int x = (home + k) % kXcds;
            const int lo = xo[x], hi = xo[x + 1];
            for (;;) {
                if (threadIdx.x == 0) s_task = lo + atomicAdd(&ctr[s * kXcds + x], 1);
                __syncthreads();
                const int i = s_task;
                // every thread holds i before s_task is rewritten, and the
                // previous task's LDS use is over
                __syncthreads();
                if (i >= hi) break;
                const int2 e = list[i];
                coop_task<RT>(P[e.x], s, e.y, smem);
            }
        }
        if (s + 1 < kStages) {
            // this stage's stores are written back before the barrier, and
            // the next stage's loads see other XCDs' stores after it
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
            cooperative_groups::this_grid().sync();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
            if (blockIdx.x == 0 && threadIdx.x < kXcds)
                __hip_atomic_store(&ctr[s * kXcds + threadIdx.x], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
}

// Merged launches: one launch per stage over every task kind of the stage
// (the per-XCD order of the fused variant, XCD-aware work-group mapping), the
// task bodies inlined behind a switch, so small kinds share a launch with
// large ones.  Mode solves of MIXED problems and of diag_waves.hip's keep the
// staged variant's launches (own_launch): their work-groups have sizes of their own, and a problem has
// to come out the same, bit for bit, whichever variant the tuner picks.  No
// waits: the launch boundaries order the stages.
template <int KIND>
__device__ __forceinline__ void merged_fft(const FftArgs &a, int L, int t, double *smem)
{
    if (L == 1) {
        unit_line_element<KIND>(a, (long long)t * 256 + threadIdx.x);
        return;
    }
    const int W = L <= 16 ? 64 : L <= 64 ? 32 : 16;
    const long long tiles = uniform_main_tiles(a.nbatch, a.lanes, a.in_batch_stride, a.out_batch_stride, W) +
                            (long long)a.xlanes * ((a.nbatch + W - 1) / W);
    if (t >= tiles) return;
    switch (L) {
    case 16: fft_tile_uniform<16, 4, 4, 64, KIND>(a, t, smem); break;
    case 32: fft_tile_uniform<32, 8, 4, 32, KIND>(a, t, smem); break;
    case 64: fft_tile_uniform<64, 8, 8, 32, KIND>(a, t, smem); break;
    case 128: fft_tile_uniform<128, 16, 8, 16, KIND>(a, t, smem); break;
    default: fft_tile_uniform<256, 16, 16, 16, KIND>(a, t, smem); break;
    }
}

template <int KIND>
__global__ __launch_bounds__(256) void batch_stage_fft(const BatchProblem *__restrict__ P,
                                                       const int2 *__restrict__ list, int pass)
{
    extern __shared__ double smem[];
    const int2 e = list[xcd_logical(blockIdx.x, gridDim.x)];
    const BatchProblem &pr = P[e.x];
    merged_fft<KIND>(pr.f[pass], pass == 0 || pass == 3 ? pr.ly : pr.lx, e.y, smem);
}

template <int RT>
__global__ __launch_bounds__(256) void batch_stage_modes(const BatchProblem *__restrict__ P,
                                                         const int2 *__restrict__ list)
{
    extern __shared__ double smem[];
    const int2 e = list[xcd_logical(blockIdx.x, gridDim.x)];
    const BatchProblem &pr = P[e.x];
    switch (pr.dkind) {
    case 0: coop_diag_t<2, RT, false>(pr.d, e.y, smem); break;
    case 2: coop_diag_t<4, RT, false>(pr.d, e.y, smem); break;
    case 3: coop_diag_t<4, RT, true>(pr.d, e.y, smem); break;
    case 4: coop_diag_t<6, RT, false>(pr.d, e.y, smem); break;
    case 5: coop_diag_t<6, RT, true>(pr.d, e.y, smem); break;
    case 6: coop_diag_t<8, RT, false>(pr.d, e.y, smem); break;
    default: coop_diag_t<8, RT, true>(pr.d, e.y, smem); break;
    }
}

// Dynamic LDS of the merged transform launches: the largest transform tile
// (the mode-solve launches take coop_lds).
constexpr size_t merged_fft_lds() { return sizeof(double) * (256 + 2) * 16; }

// Staged launches: one launch per stage and kind of task (transform length,
// or mode-solve variant), each work-group one task from a (problem, task)
// list; the launch boundaries order the stages, and every kernel inlines only
// its own body, so it gets its own register budget.
// One uniform-base tile per work-group (fft_tile_uniform: a lane block of a
// line batch, or W line batches of a face), entries in XCD-aware order.
template <int L, int R1, int R2, int W, int KIND>
__global__ __launch_bounds__(256) void batch_fft_list(const BatchProblem *__restrict__ P, const int2 *__restrict__ list,
                                                      int pass)
{
    __shared__ double tile[(L + 2) * W];
    const int2 t = list[xcd_logical(blockIdx.x, gridDim.x)];
    const FftArgs &a = P[t.x].f[pass];
    // The lists count both face tiles in the forward passes; a table filled
    // without faces simply ends here instead of reading null face pointers.
    const long long tiles = uniform_main_tiles(a.nbatch, a.lanes, a.in_batch_stride, a.out_batch_stride, W) +
                            (long long)a.xlanes * ((a.nbatch + W - 1) / W);
    if (t.y >= tiles) return;
    fft_tile_uniform<L, R1, R2, W, KIND>(a, t.y, tile);
}

// Length-1 transform passes (2-D and 1-D problems): 256 (batch, lane)
// copies per list entry.
template <int KIND>
__global__ __launch_bounds__(256) void batch_unit_list(const BatchProblem *__restrict__ P, const int2 *__restrict__ list,
                                                       int pass)
{
    const int2 t = list[blockIdx.x];
    unit_line_element<KIND>(P[t.x].f[pass], (long long)t.y * 256 + threadIdx.x);
}

__device__ __forceinline__ MixedArgs global_args(MixedArgs a)
{
    a.spec = as_global(a.spec);
    a.bc_re = as_global(a.bc_re);
    a.bc_im = as_global(a.bc_im);
    a.shift = as_global(a.shift);
    a.mu = as_global(a.mu);
    a.VinvT32 = as_global(a.VinvT32);
    a.VT32 = as_global(a.VT32);
    a.DzzTP = as_global(a.DzzTP);
    a.Dzz = as_global(a.Dzz);
    a.Dz = as_global(a.Dz);
    a.UL = as_global(a.UL);
    a.UR = as_global(a.UR);
    a.hom = as_global(a.hom);
    a.hist = as_global(a.hist);
    a.closure = as_global(a.closure);
    return a;
}

template <int NJ, int RT, bool GENERAL>
__global__ __launch_bounds__(256) void batch_diag_list(const BatchProblem *__restrict__ P, const int2 *__restrict__ list)
{
    __shared__ DiagShared<NJ, RT, GENERAL, false> sh;
    const int2 t = list[blockIdx.x];
    diag_tile<NJ, RT, GENERAL, false>(P[t.x].d, t.y, sh);
}

__device__ __forceinline__ DiagArgs global_args(DiagArgs a)
{
    a.spec = as_global(a.spec);
    a.bc_re = as_global(a.bc_re);
    a.bc_im = as_global(a.bc_im);
    a.shift = as_global(a.shift);
    a.mu = as_global(a.mu);
    a.VinvT = as_global(a.VinvT);
    a.VT = as_global(a.VT);
    a.w0 = as_global(a.w0);
    a.wN = as_global(a.wN);
    a.r0 = as_global(a.r0);
    a.rN = as_global(a.rN);
    a.hom = as_global(a.hom);
    a.closure = as_global(a.closure);
    return a;
}

// Several elements, Robin faces or periodic z at N - 2 <= 32, as a single
// solve takes them (diag_waves.hip).
template <int NJ, int WR, int RB>
__global__ __launch_bounds__(64 * NJ * WR, 4) void batch_diag_waves_list(const BatchProblem *__restrict__ P,
                                                                         const int2 *__restrict__ list)
{
    const int2 t = list[blockIdx.x];
    diag_waves_tile<NJ, WR, RB, false>(global_args(P[uniform(t.x)].d), uniform(t.y));
}

__global__ __launch_bounds__(256, 2) void batch_mixed_tile_list(const BatchProblem *__restrict__ P,
                                                                const int2 *__restrict__ list)
{
    __shared__ MixedShared<6, 32, true> sh;
    const int2 t = list[blockIdx.x];
    mixed_tile<6, 32, true>(P[t.x].m, t.y, sh);
}

// One wave per 16 columns (mixed_waves_tile), 32 rows: 48 problems of 32 to 128
// points a side 618 us, with mixed_tile's four waves a tile 877.
template <int NJ, bool GENERAL>
__global__ __launch_bounds__(64 * NJ, NJ == 6 && GENERAL ? 3 : 4) void batch_mixed_list(
    const BatchProblem *__restrict__ P, const int2 *__restrict__ list)
{
    const int2 t = list[blockIdx.x];
    mixed_waves_tile<NJ, 2, GENERAL>(global_args(P[uniform(t.x)].m), uniform(t.y));
}

}  // namespace
}  // namespace hz

using namespace hz;

// ---- host side ---------------------------------------------------------------
namespace {

// Mode-solve kinds that are launched kind by kind in every variant.
bool own_launch(int kind) { return kind >= 8; }

// One element with Dirichlet faces in DIAG form, and a grid of the z-first
// kernels (zfirst.hip): expand, filter, collect instead of the five stages.
bool z_first(const hz_plan *pl) { return pl->d.form == HZ_FORM_DIAG && pl->zf && !diag_general(pl); }

struct Variant {
    int rt;           // diag tile rows
    int fused;        // 1 one launch for the whole batch, 0 one launch per stage and task kind,
                      // 2 one launch per stage over every task kind
    const char *off;  // why the variant is refused, or null: offered to the autotuner and to hz_batch_force_variant
};

// Variants 0-3 were a persistent launch whose tasks waited on per-problem
// completion counters; its first GPU run did not finish, the cause was not
// established, and it was removed.  Variants 6 and 7 are the cooperative
// fused launch (batch_coop_kernel), switched off: variant 6 (32-row mode
// tiles) reproduced the staged results bit for bit on 512 problems and on
// periodic, 2-D and 1-D sets, but two runs did not finish -- variant 7
// (64-row tiles) on its first launch, and a batch holding MIXED plans while
// variant 6 was timed and forced -- and the cause is not established.
constexpr const char *kRemoved = "batch: variants 0-3 were removed";
constexpr const char *kCoopOff = "batch: the fused cooperative variants 6 and 7 are switched off: two GPU runs did "
                                 "not finish and the cause is not established";
const Variant kVariants[] = {{32, 1, kRemoved}, {32, 1, kRemoved}, {32, 1, kRemoved}, {64, 1, kRemoved},
                             {32, 0, nullptr},  {64, 0, nullptr},  {32, 1, kCoopOff}, {64, 1, kCoopOff},
                             {32, 2, nullptr},  {64, 2, nullptr}};
constexpr int kNumVariants = sizeof(kVariants) / sizeof(kVariants[0]);

std::mutex g_tune_mu;
std::map<std::string, int> g_tuned;  // batch shape -> variant

}  // namespace

struct hz_batch {
    std::vector<hz_plan *> plans;
    int n = 0, device = 0, cus = 0;
    hipStream_t stream = nullptr;
    hipEvent_t ev_in = nullptr, ev_out = nullptr, t0 = nullptr, t1 = nullptr;
    BatchProblem *d_probs = nullptr, *h_probs = nullptr;
    int *d_ctl = nullptr;  // [1]: error flag of the fused launch
    // staged variant: per tile height, task lists grouped by (stage, kind)
    int2 *d_list[2] = {nullptr, nullptr};
    std::vector<std::array<int, 3>> groups[2];  // {stage, kind, first}, count in next first
    // fused variant: per tile height, the same tasks in per-XCD ranges
    // (coop_order) with their bounds, the range counters, and the resident
    // work-groups per CU (0: the device cannot launch cooperatively)
    int2 *d_coop_list[2] = {nullptr, nullptr};
    int *d_coop_off[2] = {nullptr, nullptr};
    std::vector<int> h_coop_off[2];  // host copy (the merged variant's launch sizes)
    int *d_ctr = nullptr;
    int coop_wgs[2] = {0, 0};
    // z-first problems: their arguments (one entry per problem of the batch),
    // tiles and launches {stage, kind, first, count}
    ZfArgs *d_zargs = nullptr, *h_zargs = nullptr;
    int2 *d_zlist = nullptr;
    std::vector<std::array<int, 4>> zlaunches;
    bool zuse = false;
    std::vector<const void *> last;
    std::vector<unsigned> gens;  // each plan's generation when the tables were built
    std::string shape;
    int variant = -1;
    double variant_ms[kNumVariants] = {};
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
};

namespace {

int rt_index(int rt) { return rt == 64 ? 1 : 0; }

// Mode-solve tiles of a plan of that kind for DIAG tiles of `rt` rows.
int mode_tiles(const hz_plan *pl, int kind, int rt)
{
    const int rows = kind == 16 || kind == 17 ? diag_waves_rows(pl->n) : kind >= 8 ? 32 : rt;
    const int fc_per_tile = rows / (2 * pl->ne);
    const int nfc = pl->nx * pl->M;
    return (nfc + fc_per_tile - 1) / fc_per_tile;
}

int fill_problems(hz_batch *b, const double *const *f, const double *const *gl, const double *const *gr,
                  double *const *u)
{
    for (int p = 0; p < b->n; ++p) {
        hz_plan *pl = b->plans[p];
        BatchProblem &q = b->h_probs[p];
        q = BatchProblem{};
        const long long xs = pl->xs;
        q.f[0] = xy_pass_args(pl, 0, f[p], pl->spec.re, pl->spec.im, nullptr, pl->K, gl[p], gr[p], nullptr, nullptr,
                              xs);
        q.f[1] = xy_pass_args(pl, 1, nullptr, pl->spec.re, pl->spec.im, nullptr, pl->K, gl[p], gr[p], nullptr,
                              nullptr, xs);
        q.f[2] = xy_pass_args(pl, 2, nullptr, pl->spec.re, pl->spec.im, nullptr, pl->K, nullptr, nullptr, nullptr,
                              nullptr, xs);
        q.f[3] = xy_pass_args(pl, 3, nullptr, pl->spec.re, pl->spec.im, u[p], pl->K, nullptr, nullptr, nullptr,
                              nullptr, xs);
        if (z_first(pl)) b->h_zargs[p] = zf_args(pl, f[p], u[p], gl[p], gr[p]);
        if (pl->d.form == HZ_FORM_MIXED)
            q.m = mixed_args(pl);
        else
            q.d = diag_args(pl);
        q.ly = pl->ny;
        q.lx = pl->nx;
        const bool general = pl->ne > 1 || pl->d.alpha_l != 0.0 || pl->d.alpha_r != 0.0 || pl->d.periodic_z;
        const bool mixed = pl->d.form == HZ_FORM_MIXED;
        if (mixed && mixed_by_four_waves(pl->n, pl->ne, pl->nx * pl->M))
            q.dkind = 18;
        else if (general && !mixed && diag_waves_holds(pl->n, pl->ne))
            q.dkind = 16 + (pl->n > 16);
        else
            q.dkind = 2 * (diag_padded(pl->n) / 32 - 1) + (general ? 1 : 0) + (mixed ? 8 : 0);
    }
    return HZ_OK;
}

// z lanes per work-group of the batch's transform tiles of length L.
int batch_lanes(int L) { return L <= 16 ? 64 : L <= 64 ? 32 : 16; }

// Kind of a transform task: its length; of a mode-solve task: dkind.
int task_kind(const BatchProblem &q, int s) { return s == 2 ? q.dkind : (s == 0 || s == 4 ? q.ly : q.lx); }

template <int KIND>
void launch_fft_list(hipStream_t s, const BatchProblem *P, const int2 *list, int count, int L, int pass)
{
    switch (L) {
    case 1: hipLaunchKernelGGL((batch_unit_list<KIND>), dim3(count), dim3(256), 0, s, P, list, pass); break;
    case 16: hipLaunchKernelGGL((batch_fft_list<16, 4, 4, 64, KIND>), dim3(count), dim3(256), 0, s, P, list, pass); break;
    case 32: hipLaunchKernelGGL((batch_fft_list<32, 8, 4, 32, KIND>), dim3(count), dim3(256), 0, s, P, list, pass); break;
    case 64: hipLaunchKernelGGL((batch_fft_list<64, 8, 8, 32, KIND>), dim3(count), dim3(256), 0, s, P, list, pass); break;
    case 128: hipLaunchKernelGGL((batch_fft_list<128, 16, 8, 16, KIND>), dim3(count), dim3(256), 0, s, P, list, pass); break;
    default: hipLaunchKernelGGL((batch_fft_list<256, 16, 16, 16, KIND>), dim3(count), dim3(256), 0, s, P, list, pass); break;
    }
}

void launch_mixed_list(hipStream_t s, const BatchProblem *P, const int2 *list, int count, int kind)
{
    const dim3 g(count), b(128 * (kind / 2 + 1));
    switch (kind) {
    case 0: hipLaunchKernelGGL((batch_mixed_list<2, false>), g, b, 0, s, P, list); break;
    case 1: hipLaunchKernelGGL((batch_mixed_list<2, true>), g, b, 0, s, P, list); break;
    case 2: hipLaunchKernelGGL((batch_mixed_list<4, false>), g, b, 0, s, P, list); break;
    case 3: hipLaunchKernelGGL((batch_mixed_list<4, true>), g, b, 0, s, P, list); break;
    case 4: hipLaunchKernelGGL((batch_mixed_list<6, false>), g, b, 0, s, P, list); break;
    case 5: hipLaunchKernelGGL((batch_mixed_list<6, true>), g, b, 0, s, P, list); break;
    case 6: hipLaunchKernelGGL((batch_mixed_list<8, false>), g, b, 0, s, P, list); break;
    default: hipLaunchKernelGGL((batch_mixed_list<8, true>), g, b, 0, s, P, list); break;
    }
}

template <int RT>
void launch_diag_list(hipStream_t s, const BatchProblem *P, const int2 *list, int count, int kind)
{
    const dim3 g(count), b(256);
    if (kind >= 16) {
        if (kind == 18)
            hipLaunchKernelGGL(batch_mixed_tile_list, g, b, 0, s, P, list);
        else if (kind == 16)
            hipLaunchKernelGGL((batch_diag_waves_list<1, 4, 2>), g, b, 0, s, P, list);
        else
            hipLaunchKernelGGL((batch_diag_waves_list<2, 2, 2>), g, b, 0, s, P, list);
        return;
    }
    if (kind >= 8) {
        launch_mixed_list(s, P, list, count, kind - 8);
        return;
    }
    switch (kind) {
    case 0: hipLaunchKernelGGL((batch_diag_list<2, RT, false>), g, b, 0, s, P, list); break;
    case 2: hipLaunchKernelGGL((batch_diag_list<4, RT, false>), g, b, 0, s, P, list); break;
    case 3: hipLaunchKernelGGL((batch_diag_list<4, RT, true>), g, b, 0, s, P, list); break;
    case 4: hipLaunchKernelGGL((batch_diag_list<6, RT, false>), g, b, 0, s, P, list); break;
    case 5: hipLaunchKernelGGL((batch_diag_list<6, RT, true>), g, b, 0, s, P, list); break;
    case 6: hipLaunchKernelGGL((batch_diag_list<8, RT, false>), g, b, 0, s, P, list); break;
    default: hipLaunchKernelGGL((batch_diag_list<8, RT, true>), g, b, 0, s, P, list); break;
    }
}

template <int RT>
int enqueue_t(hz_batch *b, const Variant &v, hipStream_t s)
{
    const int r = rt_index(RT);
    for (const auto &z : b->zlaunches)
        if (int st = launch_zf_list(b->d_zargs, b->d_zlist + z[2], z[3], z[0], z[1], s)) return st;
    const auto &g = b->groups[r];
    if (v.fused == 2) {
        const auto &xo = b->h_coop_off[r];
        for (int st = 0; st < kStages; ++st) {
            for (size_t i = 0; st == 2 && i + 1 < g.size(); ++i)
                if (g[i][0] == 2 && own_launch(g[i][1]))
                    launch_diag_list<RT>(s, b->d_probs, b->d_list[r] + g[i][2], g[i + 1][2] - g[i][2], g[i][1]);
            const int first = xo[(size_t)st * (kXcds + 1)], count = xo[(size_t)st * (kXcds + 1) + kXcds] - first;
            if (count == 0) continue;
            const int2 *list = b->d_coop_list[r] + first;
            const dim3 grid(count), blk(256);
            const int pass = st < 2 ? st : st - 1;
            const unsigned fl = (unsigned)merged_fft_lds();
            switch (st) {
            case 0: hipLaunchKernelGGL((batch_stage_fft<FFT_R2C>), grid, blk, fl, s, b->d_probs, list, pass); break;
            case 1: hipLaunchKernelGGL((batch_stage_fft<FFT_C2C_FWD>), grid, blk, fl, s, b->d_probs, list, pass); break;
            case 2:
                hipLaunchKernelGGL((batch_stage_modes<RT>), grid, blk, (unsigned)coop_lds<RT>(), s, b->d_probs, list);
                break;
            case 3: hipLaunchKernelGGL((batch_stage_fft<FFT_C2C_INV>), grid, blk, fl, s, b->d_probs, list, pass); break;
            default: hipLaunchKernelGGL((batch_stage_fft<FFT_C2R>), grid, blk, fl, s, b->d_probs, list, pass); break;
            }
        }
        HZ_HIP(hipGetLastError());
        return HZ_OK;
    }
    if (v.fused) {
        if (b->coop_wgs[r] < 1) return set_error(HZ_ERR_UNSUPPORTED, "batch: no cooperative launch on this device");
        const BatchProblem *P = b->d_probs;
        const int2 *list = b->d_coop_list[r];
        const int *xoff = b->d_coop_off[r];
        int *ctr = b->d_ctr, *ctl = b->d_ctl;
        void *args[] = {(void *)&P, (void *)&list, (void *)&xoff, (void *)&ctr, (void *)&ctl};
        HZ_HIP(hipLaunchCooperativeKernel((const void *)batch_coop_kernel<RT>, dim3(b->coop_wgs[r] * b->cus),
                                          dim3(256), args, (unsigned)coop_lds<RT>(), s));
    } else {
        for (size_t i = 0; i + 1 < g.size(); ++i) {
            const int st = g[i][0], kind = g[i][1], first = g[i][2], count = g[i + 1][2] - first;
            if (count == 0) continue;  // e.g. only in-place length-1 passes (identities) of this kind
            const int2 *list = b->d_list[r] + first;
            const int pass = st < 2 ? st : st - 1;
            switch (st) {
            case 0: launch_fft_list<FFT_R2C>(s, b->d_probs, list, count, kind, pass); break;
            case 1: launch_fft_list<FFT_C2C_FWD>(s, b->d_probs, list, count, kind, pass); break;
            case 2: launch_diag_list<RT>(s, b->d_probs, list, count, kind); break;
            case 3: launch_fft_list<FFT_C2C_INV>(s, b->d_probs, list, count, kind, pass); break;
            default: launch_fft_list<FFT_C2R>(s, b->d_probs, list, count, kind, pass); break;
            }
        }
    }
    HZ_HIP(hipGetLastError());
    return HZ_OK;
}

// Tiles of the z-first problems, by stage and kind: 64 problems of 32 to 128
// points a side and 17 to 129 along z (317 MB) take 400 us, 600 in five stages.
// Used from one tile per CU on (16 of 32 x 32 x 17: 78 us either way; x 129 80
// against 96): on fewer, the five stages' many short work-groups fill the chip
// better.  A problem's route, and with it its low bits, so depend on the rest of
// its batch; taking the single solve's route instead runs the two halves of a
// batch one after the other (8 / 64 problems of 32 to 128 points a side 92 ->
// 133, 493 -> 633 us).
int build_zlists(hz_batch *b)
{
    int tiles = 0;
    for (const hz_plan *pl : b->plans)
        if (z_first(pl)) tiles += pl->nx * pl->ny / 64;
    b->zuse = tiles >= b->cus;
    b->zlaunches.clear();
    (void)hipFree(b->d_zlist);
    b->d_zlist = nullptr;
    if (!b->zuse) return HZ_OK;
    // {stage, launch kind} -> size -> tiles.  Within a launch, XCD x's range
    // holds the x-th eighth of every size, the larger ones first: even shares,
    // and neighbouring work-groups run the same code.
    std::map<std::pair<int, int>, std::map<int, std::vector<int2>>> by;
    for (int p = 0; p < b->n; ++p) {
        const hz_plan *pl = b->plans[p];
        if (!z_first(pl)) continue;
        for (int st = 0; st < 3; ++st) {
            auto &v = by[{st, zf_kind(pl->nx, pl->ny, pl->n, st)}][st == 1 ? -(pl->nx * 1024 + pl->ny) : -pl->NP];
            for (int t = 0, nt = zf_tasks(pl->nx, pl->ny, pl->n, st); t < nt; ++t) v.push_back(make_int2(p, t));
        }
    }
    std::vector<int2> all;
    for (auto &kv : by) {
        const size_t first = all.size();
        for (int x = 0; x < kXcds; ++x)
            for (auto &sz : kv.second) {
                const auto &v = sz.second;
                all.insert(all.end(), v.begin() + v.size() * x / kXcds, v.begin() + v.size() * (x + 1) / kXcds);
            }
        b->zlaunches.push_back({kv.first.first, kv.first.second, (int)first, (int)(all.size() - first)});
    }
    if (hipMalloc((void **)&b->d_zlist, sizeof(int2) * all.size()) != hipSuccess)
        return set_error(HZ_ERR_ALLOC, "batch allocation failed");
    HZ_HIP(hipMemcpy(b->d_zlist, all.data(), sizeof(int2) * all.size(), hipMemcpyHostToDevice));
    return HZ_OK;
}

// Task lists of the staged variant for tile height rt (problem kinds known
// from the filled problem table).
int build_lists(hz_batch *b, int rt)
{
    const int r = rt_index(rt);
    std::map<std::pair<int, int>, std::vector<int2>> by;
    for (int p = 0; p < b->n; ++p)
        for (int st = 0; st < kStages; ++st) {
            if (b->zuse && z_first(b->plans[p])) continue;
            auto &v = by[{st, task_kind(b->h_probs[p], st)}];
            int ntask = st == 2 ? mode_tiles(b->plans[p], b->h_probs[p].dkind, rt) : 0;
            if (st != 2) {  // transform passes: one entry per uniform-base tile
                // The table is filled with null buffers here, so the face
                // count is set from what hz_batch_solve always passes: both
                // faces in the forward passes (its gl, gr are never null for
                // a problem with faces), none in the inverse ones, none for
                // periodic z.  Face offsets are below nx*M.
                const FftArgs &a = b->h_probs[p].f[st < 2 ? st : st - 1];
                const bool has_faces = !b->plans[p]->d.periodic_z;
                const int L = task_kind(b->h_probs[p], st), W = batch_lanes(L);
                const int faces = st < 2 && has_faces ? 2 : 0;
                if (L == 1) {  // copies, 256 per task; the in-place x passes are identities
                    const long long total = (long long)(a.lanes + faces) * a.nbatch;
                    ntask = (st == 1 || st == 3) ? 0 : (int)((total + 255) / 256);
                    for (int t = 0; t < ntask; ++t) v.push_back(make_int2(p, t));
                    continue;
                }
                const long long lim = 1LL << 29;  // element offsets whose byte offsets fit 32 bits
                const long long m = (W - 1) + (long long)(L - 1) * std::max(a.in_point_stride, a.out_point_stride);
                if (m >= lim) return set_error(HZ_ERR_UNSUPPORTED, "batch: problem too large for a tile");
                ntask = (int)uniform_main_tiles(a.nbatch, a.lanes, a.in_batch_stride, a.out_batch_stride, W) +
                        faces * ((a.nbatch + W - 1) / W);
            }
            for (int t = 0; t < ntask; ++t) v.push_back(make_int2(p, t));
        }
    std::vector<int2> all;
    b->groups[r].clear();
    for (auto &kv : by) {  // ordered by stage, then kind
        b->groups[r].push_back({kv.first.first, kv.first.second, (int)all.size()});
        all.insert(all.end(), kv.second.begin(), kv.second.end());
    }
    b->groups[r].push_back({kStages, 0, (int)all.size()});
    (void)hipFree(b->d_list[r]);
    b->d_list[r] = nullptr;
    // (one entry more: a batch of z-first problems only has none)
    if (hipMalloc((void **)&b->d_list[r], sizeof(int2) * (all.size() + 1)) != hipSuccess)
        return set_error(HZ_ERR_ALLOC, "batch allocation failed");
    HZ_HIP(hipMemcpy(b->d_list[r], all.data(), sizeof(int2) * all.size(), hipMemcpyHostToDevice));
    // The fused variant's order: within each stage, XCD x's range holds the
    // x-th eighth of every task kind of the stage (longer transforms and
    // larger mode solves first), so the XCDs get even shares and
    // neighbouring tiles stay on one XCD's L2.
    const auto &gr = b->groups[r];
    std::vector<int2> co;
    std::vector<int> xo((size_t)kStages * (kXcds + 1), 0);
    for (int st = 0; st < kStages; ++st) {
        for (int x = 0; x < kXcds; ++x) {
            xo[(size_t)st * (kXcds + 1) + x] = (int)co.size();
            for (size_t gi = gr.size() - 1; gi-- > 0;) {
                if (gr[gi][0] != st || (st == 2 && own_launch(gr[gi][1]))) continue;
                const long long first = gr[gi][2], count = gr[gi + 1][2] - first;
                co.insert(co.end(), all.begin() + (first + count * x / kXcds),
                          all.begin() + (first + count * (x + 1) / kXcds));
            }
        }
        xo[(size_t)st * (kXcds + 1) + kXcds] = (int)co.size();
    }
    size_t own = 0;
    for (size_t gi = 0; gi + 1 < gr.size(); ++gi)
        if (gr[gi][0] == 2 && own_launch(gr[gi][1])) own += gr[gi + 1][2] - gr[gi][2];
    if (co.size() + own != all.size()) return set_error(HZ_ERR_HIP, "batch: fused task order lost tasks");
    (void)hipFree(b->d_coop_list[r]);
    (void)hipFree(b->d_coop_off[r]);
    b->d_coop_list[r] = nullptr;
    b->d_coop_off[r] = nullptr;
    if (hipMalloc((void **)&b->d_coop_list[r], sizeof(int2) * (co.size() + 1)) != hipSuccess ||
        hipMalloc((void **)&b->d_coop_off[r], sizeof(int) * xo.size()) != hipSuccess)
        return set_error(HZ_ERR_ALLOC, "batch allocation failed");
    HZ_HIP(hipMemcpy(b->d_coop_list[r], co.data(), sizeof(int2) * co.size(), hipMemcpyHostToDevice));
    HZ_HIP(hipMemcpy(b->d_coop_off[r], xo.data(), sizeof(int) * xo.size(), hipMemcpyHostToDevice));
    b->h_coop_off[r] = xo;
    return HZ_OK;
}

int enqueue(hz_batch *b, int vi, hipStream_t s)
{
    const Variant &v = kVariants[vi];
    return v.rt == 64 ? enqueue_t<64>(b, v, s) : enqueue_t<32>(b, v, s);
}

// Refill the problem table with these buffers and upload it.
int upload_problems(hz_batch *b, const double *const *f, const double *const *gl, const double *const *gr,
                    double *const *u)
{
    HZ_HIP(hipStreamSynchronize(b->stream));  // the pinned table may still be in flight
    fill_problems(b, f, gl, gr, u);
    HZ_HIP(hipMemcpyAsync(b->d_probs, b->h_probs, sizeof(BatchProblem) * b->n, hipMemcpyHostToDevice, b->stream));
    HZ_HIP(hipMemcpyAsync(b->d_zargs, b->h_zargs, sizeof(ZfArgs) * b->n, hipMemcpyHostToDevice, b->stream));
    return HZ_OK;
}

// Autotuning key of a batch: every plan's size and sweep kind.
std::string batch_shape(const std::vector<hz_plan *> &plans)
{
    std::string shape;
    for (const hz_plan *pl : plans) {
        const bool general = pl->ne > 1 || pl->d.alpha_l != 0.0 || pl->d.alpha_r != 0.0 || pl->d.periodic_z;
        shape += std::to_string(pl->nx) + "x" + std::to_string(pl->ny) + "x" + std::to_string(pl->N) + "e" +
                 std::to_string(pl->ne) + (pl->d.form == HZ_FORM_MIXED ? "m" + std::to_string(pl->sweeps) : "") +
                 (pl->d.periodic_z ? "p;" : general ? "g;" : ";");
    }
    return shape;
}

// Task lists of both tile heights from the plans as they are now (the
// mode-solve kind of a problem follows its Robin coefficients); the
// recorded graph and the uploaded table are dropped, so the next solve
// re-reads every plan.
int rebuild_lists(hz_batch *b)
{
    std::vector<const double *> nil(b->n, nullptr);
    std::vector<double *> nilo(b->n, nullptr);
    if (int st = build_zlists(b)) return st;
    for (int r = 0; r < 2; ++r) {
        fill_problems(b, nil.data(), nil.data(), nil.data(), nilo.data());
        if (int st = build_lists(b, r ? 64 : 32)) return st;
    }
    if (b->exec) (void)hipGraphExecDestroy(b->exec);
    if (b->graph) (void)hipGraphDestroy(b->graph);
    b->exec = nullptr;
    b->graph = nullptr;
    b->last.clear();
    b->gens.resize(b->n);
    for (int p = 0; p < b->n; ++p) b->gens[p] = b->plans[p]->generation;
    b->shape = batch_shape(b->plans);
    return HZ_OK;
}

// Work-groups per CU of the fused launch: as many as can be resident (at
// most 4), the condition of a cooperative launch.
template <int RT>
int coop_residency(int *wgs)
{
    *wgs = 0;
    const void *fn = (const void *)batch_coop_kernel<RT>;
    const int lds = (int)coop_lds<RT>();
    HZ_HIP(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, lds));
    int nb = 0;
    HZ_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, fn, 256, (size_t)lds));
    *wgs = std::min(nb, 4);
    return HZ_OK;
}

bool variant_usable(const hz_batch *b, int vi)
{
    const Variant &v = kVariants[vi];
    if (v.off) return false;
    if (v.fused != 1) return true;
    for (int p = 0; p < b->n; ++p)  // the fused launch has no body for the kinds with launches of their own
        if (own_launch(b->h_probs[p].dkind)) return false;
    return b->coop_wgs[rt_index(v.rt)] > 0;
}

void free_batch(hz_batch *b)
{
    if (!b) return;
    // work enqueued by hz_batch_solve may still read the tables below
    if (b->stream) (void)hipStreamSynchronize(b->stream);
    if (b->exec) (void)hipGraphExecDestroy(b->exec);
    if (b->graph) (void)hipGraphDestroy(b->graph);
    for (hipEvent_t e : {b->ev_in, b->ev_out, b->t0, b->t1})
        if (e) (void)hipEventDestroy(e);
    if (b->stream) (void)hipStreamDestroy(b->stream);
    (void)hipFree(b->d_probs);
    (void)hipHostFree(b->h_probs);
    (void)hipFree(b->d_zargs);
    (void)hipHostFree(b->h_zargs);
    (void)hipFree(b->d_zlist);
    for (int2 *l : b->d_list) (void)hipFree(l);
    for (int2 *l : b->d_coop_list) (void)hipFree(l);
    for (int *o : b->d_coop_off) (void)hipFree(o);
    (void)hipFree(b->d_ctl);
    (void)hipFree(b->d_ctr);
    delete b;
}

}  // namespace

extern "C" {

int hz_batch_create(hz_plan *const *plans, int count, hz_batch **batch)
{
    if (!plans || !batch || count < 1) return set_error(HZ_ERR_ARG, "bad argument");
    *batch = nullptr;
    int dev = 0;
    HZ_HIP(hipGetDevice(&dev));
    for (int p = 0; p < count; ++p) {
        const hz_plan *pl = plans[p];
        if (!pl) return set_error(HZ_ERR_ARG, "null plan");
        for (int q = 0; q < p; ++q)
            if (plans[q] == pl) return set_error(HZ_ERR_ARG, "a plan appears twice in the batch");
        if (pl->d.form != HZ_FORM_DIAG && pl->d.form != HZ_FORM_MIXED)
            return set_error(HZ_ERR_UNSUPPORTED, "batch: DIAG- or MIXED-form plans only");
        if (pl->device != dev) return set_error(HZ_ERR_ARG, "batch: plans on another device");
        if (pl->n > 128) return set_error(HZ_ERR_UNSUPPORTED, "batch: N-2 must be <= 128");
        if ((pl->nx != 1 && (pl->nx < 16 || pl->nx > 256)) || (pl->ny != 1 && (pl->ny < 16 || pl->ny > 256)))
            return set_error(HZ_ERR_UNSUPPORTED, "batch: nx, ny must be 1 or in [16, 256]");
        if (2 * pl->ne > 32) return set_error(HZ_ERR_UNSUPPORTED, "batch: at most 16 elements");
    }
    hz_batch *b = new hz_batch();
    b->plans.assign(plans, plans + count);
    b->n = count;
    b->device = dev;
    b->shape = batch_shape(b->plans);
    int st = HZ_OK;
    auto fail = [&](int code) {
        free_batch(b);
        return code;
    };
    if (hipDeviceGetAttribute(&b->cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || b->cus < 1)
        return fail(set_error(HZ_ERR_HIP, "cannot read the CU count"));
    if (hipStreamCreateWithFlags(&b->stream, hipStreamNonBlocking) != hipSuccess ||
        hipEventCreateWithFlags(&b->ev_in, hipEventDisableTiming) != hipSuccess ||
        hipEventCreateWithFlags(&b->ev_out, hipEventDisableTiming) != hipSuccess ||
        hipEventCreate(&b->t0) != hipSuccess || hipEventCreate(&b->t1) != hipSuccess)
        return fail(set_error(HZ_ERR_HIP, "stream/event creation failed"));
    if (hipMalloc((void **)&b->d_probs, sizeof(BatchProblem) * count) != hipSuccess ||
        hipHostMalloc((void **)&b->h_probs, sizeof(BatchProblem) * count) != hipSuccess ||
        hipMalloc((void **)&b->d_zargs, sizeof(ZfArgs) * count) != hipSuccess ||
        hipHostMalloc((void **)&b->h_zargs, sizeof(ZfArgs) * count) != hipSuccess ||
        hipMalloc((void **)&b->d_ctl, sizeof(int) * 4) != hipSuccess ||
        hipMalloc((void **)&b->d_ctr, sizeof(int) * kStages * kXcds) != hipSuccess)
        return fail(set_error(HZ_ERR_ALLOC, "batch allocation failed"));
    // hz_batch_status reads the error flag whatever ran, and the fused
    // launch expects its range counters at zero (cleared outside any graph)
    if (hipMemset(b->d_ctl, 0, sizeof(int) * 4) != hipSuccess ||
        hipMemset(b->d_ctr, 0, sizeof(int) * kStages * kXcds) != hipSuccess)
        return fail(set_error(HZ_ERR_HIP, "batch control clear failed"));
    // the merged mode-solve launch of 64-row tiles takes more than 64 KiB of dynamic LDS
    if (hipFuncSetAttribute((const void *)batch_stage_modes<64>, hipFuncAttributeMaxDynamicSharedMemorySize,
                            (int)coop_lds<64>()) != hipSuccess ||
        hipFuncSetAttribute((const void *)batch_stage_modes<32>, hipFuncAttributeMaxDynamicSharedMemorySize,
                            (int)coop_lds<32>()) != hipSuccess)
        return fail(set_error(HZ_ERR_HIP, "batch: cannot set the merged launch's LDS size"));
    int coop = 0;
    if (hipDeviceGetAttribute(&coop, hipDeviceAttributeCooperativeLaunch, dev) != hipSuccess) coop = 0;
    if (coop) {
        if ((st = coop_residency<32>(&b->coop_wgs[0])) || (st = coop_residency<64>(&b->coop_wgs[1])))
            return fail(st);
    }
    // kinds only depend on the plans: the lists are built from a table
    // filled with null buffers
    if ((st = rebuild_lists(b))) return fail(st);
    {
        std::lock_guard<std::mutex> lk(g_tune_mu);
        auto it = g_tuned.find(b->shape);
        if (it != g_tuned.end() && variant_usable(b, it->second)) b->variant = it->second;
    }
    *batch = b;
    return HZ_OK;
}

int hz_batch_solve(hz_batch *b, const double *const *f, const double *const *gl, const double *const *gr,
                   double *const *u, hz_stream_t stream)
{
    if (!b || !f || !gl || !gr || !u) return set_error(HZ_ERR_ARG, "null argument");
    for (int p = 0; p < b->n; ++p) {
        if (!f[p] || !u[p]) return set_error(HZ_ERR_ARG, "null buffer");
        if (b->plans[p]->d.periodic_z ? (gl[p] || gr[p]) : (!gl[p] || !gr[p]))
            return set_error(HZ_ERR_ARG, "face data: required without periodic z, NULL with it");
    }
    const hipStream_t cs = (hipStream_t)stream;
    int st;
    // a plan's lambda or Robin coefficients changed since the tables were
    // built (hz_plan_set_lambda / hz_plan_set_robin): rebuild them
    for (int p = 0; p < b->n; ++p)
        if (b->plans[p]->generation != b->gens[p]) {
            HZ_HIP(hipStreamSynchronize(b->stream));  // a replay may still read the old tables
            if ((st = rebuild_lists(b))) return st;
            break;
        }
    HZ_HIP(hipEventRecord(b->ev_in, cs));
    HZ_HIP(hipStreamWaitEvent(b->stream, b->ev_in, 0));
    std::vector<const void *> ptrs;
    for (int p = 0; p < b->n; ++p) {
        ptrs.push_back(f[p]);
        ptrs.push_back(gl[p]);
        ptrs.push_back(gr[p]);
        ptrs.push_back(u[p]);
    }
    if (ptrs != b->last) {
        if ((st = upload_problems(b, f, gl, gr, u))) return st;
        b->last = ptrs;
    }
    if (b->variant < 0) {
        // autotune: time every variant on these buffers (each run is a full solve)
        double best = 1e300;
        int bi = -1;
        for (int vi = 0; vi < kNumVariants; ++vi) {
            if (!variant_usable(b, vi)) continue;
            if ((st = enqueue(b, vi, b->stream))) return st;  // warm-up
            HZ_HIP(hipEventRecord(b->t0, b->stream));
            for (int r = 0; r < 3; ++r)
                if ((st = enqueue(b, vi, b->stream))) return st;
            HZ_HIP(hipEventRecord(b->t1, b->stream));
            HZ_HIP(hipEventSynchronize(b->t1));
            float ms = 0.0f;
            HZ_HIP(hipEventElapsedTime(&ms, b->t0, b->t1));
            b->variant_ms[vi] = ms / 3.0;
            if (ms < best) {
                best = ms;
                bi = vi;
            }
        }
        if (bi < 0) return set_error(HZ_ERR_UNSUPPORTED, "batch: no variant runs on this device");
        b->variant = bi;
        std::lock_guard<std::mutex> lk(g_tune_mu);
        g_tuned[b->shape] = bi;
    }
    if (kVariants[b->variant].fused == 1) {
        // one cooperative launch per solve (not recorded in a graph)
        if ((st = enqueue(b, b->variant, b->stream))) return st;
        HZ_HIP(hipEventRecord(b->ev_out, b->stream));
        HZ_HIP(hipStreamWaitEvent(cs, b->ev_out, 0));
        return HZ_OK;
    }
    if (!b->exec) {
        HZ_HIP(hipStreamBeginCapture(b->stream, hipStreamCaptureModeThreadLocal));
        st = enqueue(b, b->variant, b->stream);
        hipGraph_t g = nullptr;
        const hipError_t e = hipStreamEndCapture(b->stream, &g);
        if (st) return st;
        if (e != hipSuccess) return set_error(HZ_ERR_HIP, std::string("graph capture: ") + hipGetErrorString(e));
        b->graph = g;
        HZ_HIP(hipGraphInstantiate(&b->exec, b->graph, nullptr, nullptr, 0));
    }
    HZ_HIP(hipGraphLaunch(b->exec, b->stream));
    HZ_HIP(hipEventRecord(b->ev_out, b->stream));
    HZ_HIP(hipStreamWaitEvent(cs, b->ev_out, 0));
    return HZ_OK;
}

int hz_batch_status(hz_batch *b)
{
    if (!b) return set_error(HZ_ERR_ARG, "null argument");
    HZ_HIP(hipStreamSynchronize(b->stream));
    int flags[2] = {0, 0};
    HZ_HIP(hipMemcpy(flags, b->d_ctl, sizeof(flags), hipMemcpyDeviceToHost));
    if (flags[1]) return set_error(HZ_ERR_HIP, "batch: the fused kernel was not launched cooperatively");
    return HZ_OK;
}

int hz_batch_tuning(const hz_batch *b, int *variant, int *fused, int *tile_rows, int *wgs_per_cu,
                    double *variant_ms, int max_variants)
{
    if (!b) return set_error(HZ_ERR_ARG, "null argument");
    const int vi = b->variant;
    if (variant) *variant = vi;
    if (vi >= 0) {
        if (fused) *fused = kVariants[vi].fused;
        if (tile_rows) *tile_rows = kVariants[vi].rt;
        if (wgs_per_cu) *wgs_per_cu = kVariants[vi].fused ? b->coop_wgs[rt_index(kVariants[vi].rt)] : 0;
    }
    if (variant_ms)
        for (int i = 0; i < kNumVariants && i < max_variants; ++i) variant_ms[i] = b->variant_ms[i];
    return HZ_OK;
}

int hz_batch_force_variant(hz_batch *b, int variant)
{
    if (!b || variant < -1 || variant >= kNumVariants) return set_error(HZ_ERR_ARG, "bad variant");
    if (variant >= 0 && kVariants[variant].off) return set_error(HZ_ERR_UNSUPPORTED, kVariants[variant].off);
    if (variant >= 0 && !variant_usable(b, variant))
        return set_error(HZ_ERR_UNSUPPORTED, "batch: no cooperative launch on this device");
    if (b->exec) (void)hipGraphExecDestroy(b->exec);
    if (b->graph) (void)hipGraphDestroy(b->graph);
    b->exec = nullptr;
    b->graph = nullptr;
    b->variant = variant;
    return HZ_OK;
}

int hz_batch_destroy(hz_batch *b)
{
    free_batch(b);
    return HZ_OK;
}

int hz_solve_batched(hz_plan *const *plans, int count, const double *const *f, const double *const *gl,
                     const double *const *gr, double *const *u, hz_stream_t stream)
{
    hz_batch *b = nullptr;
    int st = hz_batch_create(plans, count, &b);
    if (st) return st;
    st = hz_batch_solve(b, f, gl, gr, u, stream);
    if (!st) st = hz_batch_status(b);
    if (!st) HZ_HIP(hipStreamSynchronize((hipStream_t)stream));
    free_batch(b);
    return st;
}

}  // extern "C"
