// GpuTlmHip.hip - C ABI of the gfx950 TLM step (include/GpuTlmHip.h).
//
// Replaces the OpenGL set-up and per-step dispatch of GpuTlm::run
// (GpuTlm.cpp:532-884 in the reference) with HIP: one stream per context,
// device-resident per-step tables, two launches per step (inject, then the
// fused scatter/connect whose extra workgroups take the monitor records; one
// where the step adds the sources itself, one for two steps of most FP32 grids)
// and no host synchronisation inside a run.
#include "tlm_context.h"

#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <exception>
#include <map>
#include <string>
#include <thread>
#include <vector>

namespace {

thread_local std::string g_create_error = "no error";

struct DevBuf
{
    void *p = nullptr;
    size_t bytes = 0;
};

} // namespace


namespace tlmi {

int fail(tlm_ctx *c, int code, const std::string &msg)
{
    if (c)
        c->err = msg;
    else
        g_create_error = msg;
    return code;
}



// Launch shape: a wave task is one 64-cell strip of a z-slab marched over
// zc slabs (tuning.planes; 0 picks zc for about 64K tasks). Task groups of
// block_waves tasks go to workgroups; tuning.grid_blocks > 0 caps the grid
// (persistent workgroups walking their XCD's range of groups).
int step_occupancy(const tlm_ctx *c);

void choose_shape(tlm_ctx *c)
{
    c->strips = (int)(c->Pp / tlm::kWave);
    if (c->tune.planes > 0)
        c->zc = std::min(c->tune.planes, c->nz);
    else
    {
        const long long target = 65536;
        int nch = (int)std::max(1LL, std::min<long long>(c->nz, target / c->strips));
        c->zc = (c->nz + nch - 1) / nch;
    }
    c->nzc = (c->nz + c->zc - 1) / c->zc;
    c->tasks = c->strips * c->nzc;
    // waves per workgroup: 4, or 2 when the step runs under the occupancy cap
    // (ms a launch at 4 / 2 / 1: 512^3 64 boxes 2.535 / 2.527 / 2.522, 384^3
    // 1.069 / 1.057 / 1.059, 512^3 free space 2.180 / 2.180 / 2.183; uncapped
    // 256^3 8 boxes 0.282 / 0.282 / 0.285)
    const int auto_waves = c->pf == TLM_PULSE_F32 && step_occupancy(c) > 0 ? 2 : 4;
    c->wpb = std::max(1, std::min(4, c->tune.block_waves > 0 ? c->tune.block_waves : auto_waves));
    c->groups = (c->tasks + c->wpb - 1) / c->wpb;
    c->blocks = c->tune.grid_blocks > 0 ? std::min(c->groups, c->tune.grid_blocks) : c->groups;
    // One workgroup per group: XCD x takes chunks x, x + 8, ... of half a
    // z-slab's (or z-chunk's) groups, so that each XCD's share holds an even
    // sample of the grid's depth and no XCD is left with most of its
    // dielectric blocks (the step ends with the last XCD); a chunk's groups
    // stay on one XCD, so the slots that two waves share (strip seams, rows)
    // meet in one L2. A persistent grid keeps contiguous ranges.
    c->xchunk = 0;
    if (c->tune.grid_blocks <= 0)
    {
        c->xchunk = std::max(1, std::min(c->strips / c->wpb / 2, (c->groups + 7) / 8));
        c->blocks = 8 * tlm::xcd_chunk_map(c->groups, c->xchunk).cpx;
    }
}

// Energy partials that one workgroup adds up in a launch; more are added in two.
constexpr long long kEnergyOneStage = 32768;

// One energy partial per 64-cell block, whatever the launch (block_energy).
size_t energy_parts(const tlm_ctx *c)
{
    return (size_t)c->P / tlm::kWave;
}

// ---- two steps a launch (k_step2) ----

// Tile of a workgroup (one 64-cell block per wave and `cells`): C blocks per
// wave, tb blocks of the tile, hb = ceil(nx / 64) blocks of rim on either
// side, marched over zc slabs. Measured on 20 grids (us a step, tiles of one
// / two blocks per wave): below ~6 M cells one block per wave leaves more
// workgroups and shorter slabs (96^3 12.0 / 13.4, 128^3 21.2 / 22.5), above
// it two reread less of the rim (256^3 182 / 171, 384^3 966 / 612). Few
// blocks a tile where the grid is too small to fill the chip otherwise (24^3
// 2.98 at 1 block, 3.24 at 8; 64^3 5.5 at 4, 6.1 at 8). A slab count that
// gives every CU the same number of workgroups beats a longer march (160^3:
// 46.7 at 250 workgroups of 32 slabs, 56 at 400 of 24).
// The rim is 2 hb blocks of step n done twice: a tile of tb >= 8 blocks pays
// up to hb = 12 (768 x 128 x 256: 318 against 414 us a step for two k_step
// launches), one of 2 blocks at hb = 15 does not (606 against 263 us), so
// grids wider than 768 cells keep single steps. Over 100 grids of 330, 513, 600,
// 700 and 768 cells of width, 3 to 768 rows and 3 to 768 slabs, with and without
// stubs, a pair takes 0.54 to 0.96 of the single steps' time in all but two (513 x
// 8 x 300 with stubs 1.02, 700 x 16 x 16 with stubs 1.04).
constexpr int kPairMaxRim = 12, kPairWaves = 16, kCus = 256;
void choose_pair(tlm_ctx *c)
{
    auto &p = c->pair;
    p.hb = (c->nx + tlm::kWave - 1) / tlm::kWave;
    p.ok = c->pf == TLM_PULSE_F32 && p.hb <= kPairMaxRim;
    if (!p.ok)
        return;
    const long long ncell = (long long)c->nx * c->ny * c->nz;
    p.cells = ncell >= (6LL << 20) || p.hb > 4 ? 2 : 1;
    if (p.cells == 2)
        p.tb = std::min(16, 2 * (kPairWaves - p.hb));
    else
        p.tb = ncell < 50000 ? 2 : ncell < 400000 ? 4 : 8;
    p.tb = std::min(p.tb, (c->strips + p.cells - 1) / p.cells * p.cells);
    p.ntile = (c->strips + p.tb - 1) / p.tb;
    if (p.ntile == 1)
        p.hb = 0; // the tile is the slab
    p.nt = (p.tb + 2 * p.hb) / p.cells * tlm::kWave;
    // slabs per tile: the fewest slab iterations (zc and the two beside them)
    // over the rounds that the CUs take
    long long best = 0;
    for (int most = std::min(64, c->nz); most >= 1; --most)
    {
        const int nzc = (c->nz + most - 1) / most, z = (c->nz + nzc - 1) / nzc;
        const long long cost = ((long long)p.ntile * ((c->nz + z - 1) / z) + kCus - 1) / kCus * (z + 2);
        if (best == 0 || cost < best)
        {
            best = cost;
            p.zc = z;
        }
    }
    p.groups = p.ntile * ((c->nz + p.zc - 1) / p.zc);
    // equal shares for the XCDs: 8 m chunks of at most a slab's tiles (chunks
    // of a whole slab left XCDs idle: 192^3 96 against 80 us a step)
    const int m = (p.groups + 8 * p.ntile - 1) / (8 * p.ntile);
    p.chunk = (p.groups + 8 * m - 1) / (8 * m);
    p.blocks = 8 * tlm::xcd_chunk_map(p.groups, p.chunk).cpx;
}

// The fused step launch; nmon > 0 appends the workgroups that take the
// step's monitor records. With events e0 / e1 the launch carries them as its
// own start / end timestamps (hipExtLaunchKernel): a marker recorded on the
// stream between two kernels would add a gap of ~5 us before and after the
// step, which hipEventRecord on either side of it measured.
// Dynamic LDS per workgroup that holds the step kernel to `occ` waves per
// SIMD (workgroups of wpb waves, 160 KB of LDS per CU): the kernel uses no
// LDS, the share only limits how many of its workgroups a CU takes. On
// large FP32 grids 5 waves per SIMD keep HBM as busy as more do and contend
// less (512^3 steps: plain air 2.219 against 2.275 ms, 64 dielectric boxes
// 2.684 against 2.745 ms); at 256^3 a cap costs 1 % and 16-bit steps gain
// nothing, so those run uncapped.
constexpr int kLdsPerCu = 160 * 1024;
int lds_share(int occ, int wpb)
{
    if (occ <= 0)
        return 0;
    const int wg = std::max(1, occ * 4 / wpb); // workgroups per CU
    return (kLdsPerCu / wg) & ~1023;           // (wg + 1) shares no longer fit
}

constexpr long long kOccCapCells = 32LL << 20;
int step_occupancy(const tlm_ctx *c)
{
    if (c->tune.occupancy >= 0)
        return c->tune.occupancy;
    return c->pf == TLM_PULSE_F32 && (long long)c->nx * c->ny * c->nz >= kOccCapCells ? 5 : 0;
}

template <bool S, bool E, int PF>
void launch_fused(tlm_ctx *c, const tlm::StepArgs &a, const tlm::MonitorArgs &m, int nmon,
                  hipEvent_t e0, hipEvent_t e1)
{
    const int bt = c->wpb * tlm::kWave;
    const int mon_blocks = nmon > 0 ? (nmon + bt - 1) / bt : 0;
    dim3 grid(c->blocks + mon_blocks), block(bt);
    const int shm = lds_share(step_occupancy(c), c->wpb);
    // automatic: non-temporal pulse stores when the grid has stub cells
    // (faster there by 1-3 %; slower by 3-4 % in plain air)
    const bool nt = c->tune.nontemporal == 1 || (c->tune.nontemporal == 2 && c->stubs);
    auto go = [&](auto kern) {
        if (e0)
            hipExtLaunchKernelGGL(kern, grid, block, shm, c->stream, e0, e1, 0, a, m, c->blocks);
        else
            hipLaunchKernelGGL(kern, grid, block, shm, c->stream, a, m, c->blocks);
    };
    if (PF != tlm::PF_F32)
        go(tlm::k_step<S, E, false, PF>);
    else if (a.fold.ninj > 0)
        nt ? go(tlm::k_step<S, E, true, PF, true>) : go(tlm::k_step<S, E, false, PF, true>);
    else
        nt ? go(tlm::k_step<S, E, true, PF>) : go(tlm::k_step<S, E, false, PF>);
}

template <int PF>
void launch_pf(tlm_ctx *c, const tlm::StepArgs &a, bool energy, const tlm::MonitorArgs &m, int nmon,
               hipEvent_t e0, hipEvent_t e1)
{
    if (c->stubs)
        energy ? launch_fused<true, true, PF>(c, a, m, nmon, e0, e1)
               : launch_fused<true, false, PF>(c, a, m, nmon, e0, e1);
    else
        energy ? launch_fused<false, true, PF>(c, a, m, nmon, e0, e1)
               : launch_fused<false, false, PF>(c, a, m, nmon, e0, e1);
}


// FP32 contexts with a few source cells may add them inside the step
// instead of k_inject. That saves the injection launch: 64^3 free space 7.2
// against 10.6 us a step, 128^3 dielectric boxes 40.9 against 44.0 us. The
// stub kernel compiled with the folded code takes fewer registers, which
// lets more of its waves in: uncapped that is slower on mid-size grids
// (256^3 boxes: 0.2859 against 0.2826 ms a launch), under the occupancy cap
// of large grids it is faster (384^3 boxes 1.019 against 1.026 ms, 512^3
// 2.558 against 2.569 ms, the injection launch saved on top). So by default
// grids with stub cells fold up to kFoldAutoCells cells or when the step
// runs capped, grids without stub cells at any size (512^3 free space:
// equal). tuning.fold: 0 never, 1 always, 2 by that rule.
constexpr long long kFoldAutoCells = 4LL << 20;
bool fold_active(const tlm_ctx *c)
{
    if (c->pf != TLM_PULSE_F32 || c->nuniq <= 0 || c->nuniq > tlm::kFoldMax)
        return false;
    if (c->tune.fold == 1)
        return true;
    return c->tune.fold == 2 && (!c->stubs || (long long)c->nx * c->ny * c->nz <= kFoldAutoCells ||
                                 step_occupancy(c) > 0);
}

void mark_fold(tlm_ctx *c, hipStream_t s)
{
    if (c->fold_marked)
        return;
    hipLaunchKernelGGL(tlm::k_mark_fold, dim3(1), dim3(64), 0, s, c->ucell, c->nuniq, c->uair, c->code);
    c->fold_marked = true;
}

tlm::Fold fold_at(const tlm_ctx *c, int n)
{
    tlm::Fold f;
    f.cell = c->ucell;
    f.beg = c->ubeg;
    f.pol = c->spol;
    f.amp = c->samp;
    f.ninj = c->nuniq;
    f.sv = c->sv_host[n];
    return f;
}
tlm::Fold fold_of(const tlm_ctx *c, int n)
{
    return fold_active(c) ? fold_at(c, n) : tlm::Fold();
}

// last: of a run; before any other step k_plan_inject takes the 16-bit slab maxima.
int launch_step(tlm_ctx *c, int n, bool last, const tlm::MonitorArgs &m, int nmon, hipEvent_t e0, hipEvent_t e1)
{
    const bool energy = c->every > 0 && (n % c->every) == 0;
    tlm::StepArgs a;
    a.A = c->A;
    a.B = c->B;
    a.Vs = c->Vs;
    a.code = c->code;
    a.uair = c->uair;
    a.props = c->props;
    a.epart = c->epart;
    a.slab = c->slab;
    a.dsc = nullptr;
    a.esc = nullptr;
    a.mpart = c->mpart;
    if (c->pf != TLM_PULSE_F32)
    {
        const int cur = scale_buf(c, n);
        a.dsc = c->scl[cur];
        a.esc = c->iscl[cur ^ 1];
    }
    a.nx = c->nx;
    a.ny = c->ny;
    a.nz = c->nz;
    a.nxy = (int)c->nxy;
    a.Pp = c->Pp;
    a.P = c->P;
    a.PB = c->PB;
    a.h0 = c->h0;
    a.h1 = c->h1;
    a.strips = c->strips;
    a.zc = c->zc;
    a.nzc = c->nzc;
    a.tasks = c->tasks;
    a.groups = c->groups;
    a.rho = c->rho;
    a.nmat = c->nmat;
    a.mstrips = tlm::magic_div((unsigned)c->strips);
    a.mPp = tlm::magic_div((unsigned)c->Pp);
    a.mnx = tlm::magic_div((unsigned)c->nx);
    a.xm = c->xchunk > 0 ? tlm::xcd_chunk_map(c->groups, c->xchunk) : tlm::xcd_map(c->blocks, c->groups);
    a.fold = fold_of(c, n);
    if (c->pf == TLM_PULSE_F16)
        launch_pf<tlm::PF_F16>(c, a, energy, m, nmon, e0, e1);
    else if (c->pf == TLM_PULSE_BF16)
        launch_pf<tlm::PF_BF16>(c, a, energy, m, nmon, e0, e1);
    else
        launch_pf<tlm::PF_F32>(c, a, energy, m, nmon, e0, e1);
    if (last && c->pf != TLM_PULSE_F32)
        hipLaunchKernelGGL(tlm::k_slab_max, dim3(c->nz), dim3(256), 0, c->stream, c->mpart,
                           c->strips, c->mreg);
    return TLM_OK;
}

// Whether the context's sources can be added in a pair of steps, and whether a
// pair is worth it with its monitors. A record of step n+1 takes the loads and
// scatters of seven cells (PairPulses), which costs more than the pair saves
// where most of the work are records. Per cell a face costs most when it lies
// beside others along x (a single step's loads are then whole lines), a face
// of the Huygens box less, a probe anywhere in the grid more; below 16384 faces the
// saved launch is worth more than any of them. Us a step, single / pairs:
//   PEC plates along x and y, 128^3 with 0.05, 0.06, 0.13, 0.5 faces a cell
//   31.6 / 31.0, 31.5 / 34.6, 32.0 / 50.0, 42.2 / 148; 48^3 with 0.13 and
//   0.17 6.0 / 5.3 and 6.0 / 6.7, 32^3 with 0.5 5.5 / 4.5;
//   scattered PEC cells, 128^3 with 0.06, 0.12, 0.28: 54.1 / 41.6, 62.2 / 52.4,
//   84.5 / 90.4;
//   a Huygens box, 64^3 with 0.07 and 96^3 with 0.05 11.3 / 8.6 and 22.0 / 18.6;
//   scattered probes, 128^3 with 0.015, 0.02 and 0.03 39.0 / 34.9, 41.8 / 40.2
//   and 46.7 / 52.1.
bool pair_suits(const tlm_ctx *c)
{
    const long long ncell = (long long)c->nx * c->ny * c->nz;
    return c->nuniq <= tlm::kFoldMax &&
           5LL * c->nf + 3LL * c->nh + 12LL * c->npr <= std::max(5 * 16384LL, ncell / 4);
}

// Whether pairs of steps may run as one launch: FP32 pulses, the sources and
// records few enough (pair_suits), the launch shape automatic (a
// caller's own shape is for k_step).
bool pair_active(const tlm_ctx *c)
{
    static const tlm_tuning automatic = tlm_ctx().tune;
    return c->pair.ok && !c->pair_refused && pair_suits(c) && std::memcmp(&c->tune, &automatic, sizeof(automatic)) == 0;
}

// Whether steps n and n+1 may be one pair: the energy, the cut plane and the
// frames are taken from pulses in memory, so of a pair only step n has them.
bool pair_ok(const tlm_ctx *c, int n, int end)
{
    return n + 1 < end && !(c->every > 0 && (n + 1) % c->every == 0) &&
           !(c->pa >= 0 && (n + 1) % 2 == 0) &&
           !(c->frame_every > 0 && (n % c->frame_every == 0 || (n + 1) % c->frame_every == 0));
}

// The kernel for the context's tile, with its LDS.
struct PairKernel
{
    const void *f;
    int lds;
};
template <bool S, bool E> PairKernel pair_kernel_of(const tlm_ctx *c)
{
    // an id is a byte: at most 254 dielectrics
    constexpr int nmat = S ? 254 : 0;
    if (c->pair.cells == 2)
        return {(const void *)tlm::k_step2<S, E, 2, 1024>, tlm::pair_lds<2, 1024>(nmat)};
    if (c->pair.nt <= 256)
        return {(const void *)tlm::k_step2<S, E, 1, 256>, tlm::pair_lds<1, 256>(nmat)};
    if (c->pair.nt <= 512)
        return {(const void *)tlm::k_step2<S, E, 1, 512>, tlm::pair_lds<1, 512>(nmat)};
    return {(const void *)tlm::k_step2<S, E, 1, 1024>, tlm::pair_lds<1, 1024>(nmat)};
}
PairKernel pair_kernel(const tlm_ctx *c, bool energy)
{
    if (c->stubs)
        return energy ? pair_kernel_of<true, true>(c) : pair_kernel_of<true, false>(c);
    return energy ? pair_kernel_of<false, true>(c) : pair_kernel_of<false, false>(c);
}

// Steps since the upload from which on it pays to prepare for pairs. That takes
// 15 us or, with the allocation of a large buffer, 30; a pair of a small grid
// saves 3 (8^3: the first run of 1, 4 and 16 steps 19, 32 and 83 us in single
// steps, 35, 42 and 75 with pairs from the first on; 64^3 22, 47, 142 and 49, 66,
// 148). From 3 M cells on it takes less than the first pair saves (first run of 2
// steps 162^3 225 us in single steps, 187 as a pair, 256^3 755 and 530; 128^3 85
// and 111).
long long pair_first(const tlm_ctx *c)
{
    return (long long)c->nx * c->ny * c->nz < (3LL << 20) ? 8 : 2;
}

// First pair after an upload: the second stub buffer and the kernels' LDS
// limit. The buffer starts as a copy: no step touches the stubs of the 32-cell
// halves of a block without a dielectric cell, and a caller may have uploaded
// some there, which both buffers then hold for good. A context without
// room for the buffer (it takes at most a quarter of what is free) keeps
// single steps until the next upload.
int prepare_pair(tlm_ctx *c)
{
    c->pair_ready = true;
    c->pair_refused = true;
    for (bool energy : {false, true})
    {
        const PairKernel k = pair_kernel(c, energy);
        if (k.lds > kLdsPerCu || hipFuncSetAttribute(k.f, hipFuncAttributeMaxDynamicSharedMemorySize, k.lds) != hipSuccess)
        {
            (void)hipGetLastError();
            return TLM_OK;
        }
    }
    const size_t n = (size_t)c->P * 3;
    if (c->stubs && !c->Vs2)
    {
        size_t fr = 0, tot = 0;
        if (hipMemGetInfo(&fr, &tot) != hipSuccess || n * sizeof(float) > fr / 4 ||
            hipMalloc((void **)&c->Vs2, n * sizeof(float)) != hipSuccess)
        {
            (void)hipGetLastError();
            c->Vs2 = nullptr;
            return TLM_OK;
        }
        c->owned.push_back(c->Vs2);
    }
    if (c->stubs)
        HIPCHK(c, hipMemcpyAsync(c->Vs2, c->Vs, n * sizeof(float), hipMemcpyDeviceToDevice, c->stream));
    c->pair_refused = false;
    return TLM_OK;
}

int launch_pair(tlm_ctx *c, int n, const tlm::MonitorArgs &m0, hipEvent_t e0, hipEvent_t e1)
{
    tlm::PairArgs a = {};
    a.A = c->A;
    a.B = c->B;
    a.Vs = c->Vs;
    a.Vs2 = c->Vs2;
    a.code = c->code;
    a.uair = c->uair;
    a.props = c->props;
    a.epart = c->epart;
    a.nx = c->nx;
    a.ny = c->ny;
    a.nz = c->nz;
    a.Pp = c->Pp;
    a.rho = c->rho;
    a.nmat = std::min(c->nmat, 254);
    a.strips = c->strips;
    a.tb = c->pair.tb;
    a.hb = c->pair.hb;
    a.ntile = c->pair.ntile;
    a.zc = c->pair.zc;
    a.xm = tlm::xcd_chunk_map(c->pair.groups, c->pair.chunk);
    a.mPp = tlm::magic_div((unsigned)c->Pp);
    a.mnx = tlm::magic_div((unsigned)c->nx);
    if (c->nuniq > 0)
    {
        a.fold = fold_at(c, n);
        a.sv1 = c->sv_host[n + 1];
    }
    tlm::MonitorArgs m = m0;
    m.pv.fold = a.fold;
    const int wpb = c->pair.nt / tlm::kWave;
    int mon_from = c->pair.blocks, mon_plane = (tlm::pair_face_waves(m) + m.np + wpb - 1) / wpb;
    dim3 grid(mon_from + mon_plane + (m.pn + c->pair.nt - 1) / c->pair.nt), block(c->pair.nt);
    const PairKernel k = pair_kernel(c, c->every > 0 && (n % c->every) == 0);
    void *args[] = {&a, &m, &mon_from, &mon_plane};
    if (e0)
        HIPCHK(c, hipExtLaunchKernel(k.f, grid, block, args, k.lds, c->stream, e0, e1, 0));
    else
        HIPCHK(c, hipLaunchKernel(k.f, grid, block, args, k.lds, c->stream));
    std::swap(c->Vs, c->Vs2);
    return TLM_OK;
}

void queue_probe_dft(tlm_ctx *c, int n0, int n1, hipStream_t s)
{
    if (c->npr <= 0 || c->nfreq <= 0 || n1 <= n0)
        return;
    const int tot = c->npr * 3 * c->nfreq, b = 128;
    hipLaunchKernelGGL(tlm::k_probe_dft, dim3((tot + b - 1) / b), dim3(b), 0, s, c->prrec, c->npr,
                       c->ctab, c->stab, c->nfreq, n0, n1, c->dft_re, c->dft_im);
    c->dft_done = n1;
}

tlm::PulseView pulse_view(const tlm_ctx *c, int n)
{
    tlm::PulseView v;
    v.base = c->A;
    v.PB = c->PB;
    v.Pp = c->Pp;
    v.mPp = tlm::magic_div((unsigned)c->Pp);
    v.pf = c->pf;
    v.slab = c->slab;
    v.h0 = c->h0;
    v.h1 = c->h1;
    v.sc = nullptr;
    v.isc = nullptr;
    if (c->pf != TLM_PULSE_F32)
    {
        const int cur = scale_buf(c, n);
        v.sc = c->scl[cur];
        v.isc = c->iscl[cur];
    }
    return v;
}


// kernel_every > 0: the step launches of the steps i = 0, k, 2k, ... of the
// block carry timing events; their summed duration goes to *ms_kernel, the
// number of steps they took to *nkernel.
int queue_steps(tlm_ctx *c, int step0, int nsteps, int kernel_every, float *ms_kernel, int *nkernel)
{
    if (c->batch)
        return fail(c, TLM_ERR_STATE, "context is a batch member (tlm_batch_remove it first)");
    if (!c->uploaded)
        return fail(c, TLM_ERR_STATE, "tlm_run before tlm_upload");
    if (nsteps < 0 || step0 < 0)
        return fail(c, TLM_ERR_ARG, "negative step range");
    if (nsteps == 0)
        return TLM_OK;
    if (!c->sv || step0 + nsteps > c->nsteps)
        return fail(c, TLM_ERR_STATE, "step range exceeds the schedule set by tlm_set_schedule");
    HIPCHK(c, hipSetDevice(c->dev));
    if (c->pf != TLM_PULSE_F32)
    {
        if (!c->materialized)
        {
            int rc = materialize(c, step0);
            if (rc)
                return rc;
        }
        else if (step0 != c->next_step)
            return fail(c, TLM_ERR_STATE, "16-bit pulse storage runs contiguous step blocks");
    }
    const bool fold = fold_active(c);
    if (pair_active(c) && !c->pair_ready && c->launches + c->pairs + nsteps >= pair_first(c))
    {
        int rc = prepare_pair(c);
        if (rc)
            return rc;
    }
    const bool pairs = pair_active(c) && c->pair_ready;
    if (fold || (pairs && c->nuniq > 0))
        mark_fold(c, c->stream);
    const int nmon0 = c->nf + c->nh + c->np + c->npr;
    const bool time_kernel = kernel_every > 0;
    const int ntimed = time_kernel ? (nsteps + kernel_every - 1) / kernel_every : 0;
    if (time_kernel)
    {
        // the sampled launches carry a start and an end event; no host wait
        // inside the loop
        while ((int)c->kev.size() < 2 * ntimed)
        {
            hipEvent_t ev;
            HIPCHK(c, hipEventCreate(&ev));
            c->kev.push_back(ev);
        }
    }
    const int end = step0 + nsteps;
    int per = 1; // steps of the launch
    int nev = 0, timed_steps = 0; // timed launches and their steps
    for (int n = step0; n < end; n += per)
    {
        per = pairs && pair_ok(c, n, end) ? 2 : 1;
        const tlm::PulseView pv = pulse_view(c, n);
        tlm::PlanArgs pl = {};
        if (c->pf != TLM_PULSE_F32)
        {
            const int cur = scale_buf(c, n);
            pl.nz = c->nz;
            pl.mreg = c->mreg;
            pl.Q = c->qinj;
            pl.slab = c->slab;
            pl.sv = c->sv;
            pl.n = n;
            pl.nsteps = c->nsteps;
            pl.rp = std::max(1.0f, std::fabs(c->rho));
            pl.fmax = format_max(c->pf);
            pl.isc_cur = c->iscl[cur];
            pl.sc_next = c->scl[cur ^ 1];
            pl.isc_next = c->iscl[cur ^ 1];
            pl.flag = c->flag;
        }
        if (pl.nz > 0 && n > step0)
        {
            const int np = (c->nz + tlm::kPlanSlabs - 1) / tlm::kPlanSlabs, g = (c->nuniq + 255) / 256;
            hipLaunchKernelGGL(tlm::k_plan_inject, dim3(np + g), dim3(256), 0, c->stream, pv, c->ucell, c->ubeg,
                               c->spol, c->samp, c->nuniq, c->sv, n, pl, c->mpart, c->strips, c->mreg, np);
        }
        else if ((fold || per == 2 ? 0 : c->nuniq) + pl.nz > 0)
        {
            int b = 128, g = (c->nuniq + pl.nz + b - 1) / b;
            hipLaunchKernelGGL(tlm::k_inject, dim3(g), dim3(b), 0, c->stream, pv, c->ucell,
                               c->ubeg, c->spol, c->samp, c->nuniq, c->sv, n, pl);
        }
        const bool plane_now = c->pa >= 0 && (n % 2) == 0;
        const int pn = plane_now ? c->pn1 * c->pn2 : 0;
        const int nmon = nmon0 + pn;
        tlm::MonitorArgs m = {};
        if (nmon > 0)
        {
            m.pn = pn;
            m.pa = c->pa;
            m.pidx = c->pidx;
            m.pn1 = c->pn1;
            m.pn2 = c->pn2;
            m.nx = c->nx;
            m.ny = c->ny;
            m.Pp = c->Pp;
            m.code = c->code;
            m.plane = c->plane;
            m.pv = pv;
            m.pv.fold = fold_of(c, n);
            m.n = n;
            m.settle = c->settle;
            m.cph = c->cph;
            m.sph = c->sph;
            m.nf = c->nf;
            m.fcell = c->fcell;
            m.faxis = c->faxis;
            m.js_inst = c->js_inst;
            m.js_dft4 = c->js_dft4;
            m.nh = c->nh;
            m.hcell = c->hcell;
            m.haxis = c->haxis;
            m.huy8 = c->huy8;
            m.np = c->np;
            m.pcells = c->pcells;
            m.poff = c->poff;
            m.ppol = c->ppol;
            m.ploop = c->ploop;
            m.prec = c->prec;
            m.npr = c->npr;
            m.prcell = c->prcell;
            m.inv_dl = c->inv_dl;
            m.prrec = c->prrec;
            if (plane_now)
                c->plane_step = n;
        }
        // the monitor records of step n run in the step launch's extra workgroups
        // a launch is timed if one of its steps is among the sampled ones
        const int ti = n - step0;
        const bool timed = time_kernel && (ti + per - 1) / kernel_every * kernel_every >= ti;
        hipEvent_t e0 = nullptr, e1 = nullptr;
        if (timed)
        {
            e0 = c->kev[2 * nev];
            e1 = c->kev[2 * nev + 1];
            ++nev;
            timed_steps += per;
        }
        if (per == 2)
        {
            int rc = launch_pair(c, n, m, e0, e1);
            if (rc)
                return rc;
        }
        else
            launch_step(c, n, n + 1 == end, m, nmon, e0, e1);
        ++c->launches;
        c->pairs += per == 2;
        if (c->frame_every > 0 && (n % c->frame_every) == 0 &&
            (int)c->frame_steps.size() < c->frame_max)
        {
            // TlmSolver.cpp:747-763: the frame keeps |Js| of this step and the latest plane
            const size_t f = c->frame_steps.size();
            if (c->nf > 0)
                HIPCHK(c, hipMemcpyAsync(c->frame_js + f * c->nf, c->js_inst, c->nf * sizeof(float),
                                         hipMemcpyDeviceToDevice, c->stream));
            const size_t np2 = (size_t)c->pn1 * c->pn2;
            if (c->pa >= 0 && c->plane_step >= 0)
                HIPCHK(c, hipMemcpyAsync(c->frame_plane + f * np2, c->plane, np2 * sizeof(float),
                                         hipMemcpyDeviceToDevice, c->stream));
            c->frame_steps.push_back(n);
            c->frame_plane_step.push_back(c->pa >= 0 ? c->plane_step : -1);
        }
        if (c->every > 0 && (n % c->every) == 0)
        {
            const int idx = n / c->every;
            const long long np = (long long)energy_parts(c);
            if (np > kEnergyOneStage)
            {
                // two stages: 1024 fixed chunks, then one block
                const long long chunk = (np + 1023) / 1024;
                const int nb = (int)((np + chunk - 1) / chunk);
                hipLaunchKernelGGL(tlm::k_energy_chunks, dim3(nb), dim3(tlm::kEnergyChunk), 0, c->stream,
                                   c->epart, np, chunk, c->epart2);
                hipLaunchKernelGGL(tlm::k_energy_reduce, dim3(1), dim3(tlm::kEnergyReduce), 0, c->stream,
                                   c->epart2, nb, c->energy + idx);
            }
            else
                hipLaunchKernelGGL(tlm::k_energy_reduce, dim3(1), dim3(tlm::kEnergyReduce), 0, c->stream,
                                   c->epart, (int)np, c->energy + idx);
            if ((int)c->energy_steps.size() <= idx)
                c->energy_steps.resize(idx + 1, -1);
            c->energy_steps[idx] = n;
        }
        std::swap(c->A, c->B);
    }
    HIPCHK(c, hipGetLastError());
    // running probe DFT over the newly recorded steps, in step order
    if (c->npr > 0 && c->nfreq > 0)
    {
        if (step0 != c->dft_done)
            return fail(c, TLM_ERR_STATE, "probe DFT needs contiguous step blocks from step 0");
        queue_probe_dft(c, step0, step0 + nsteps, c->stream);
    }
    c->steps_run_hi = std::max(c->steps_run_hi, step0 + nsteps);
    c->next_step = step0 + nsteps;
    if (time_kernel && ms_kernel)
    {
        float kern_ms = 0.f;
        HIPCHK(c, hipEventSynchronize(c->kev[2 * nev - 1]));
        for (int s = 0; s < nev; ++s)
        {
            float ms = 0.f;
            HIPCHK(c, hipEventElapsedTime(&ms, c->kev[2 * s], c->kev[2 * s + 1]));
            kern_ms += ms;
        }
        *ms_kernel = kern_ms;
        if (nkernel)
            *nkernel = timed_steps;
        c->timed_launches = nev;
        c->timed_pairs = timed_steps - nev;
    }
    HIPCHK(c, hipGetLastError());
    return TLM_OK;
}

// Threads that move host memory: a first write to fresh memory costs more in
// page faults (45 us a MB) than the copy itself, and they are taken side by
// side. Their pinned memory stays at 8 MB, above which it takes 2 to 4 ms to
// make or give back in some processes (reading 64^3 cells 0.65 ms with four
// threads of 2 MB, 2.5 with six or eight; 157^3 8.1, 7.2 with six).
constexpr int kHostThreads = 4;
constexpr size_t kHostChunk = (size_t)2 << 20; // bytes per turn of a thread

// Runs work(w) on up to n <= kHostThreads threads, w = 0 on the calling one;
// fewer where the system gives no more threads or memory for them (no exception
// leaves an entry point of the library). work must finish the job whichever of
// them run.
template <class F> void on_threads(int n, const F &work)
{
    std::thread t[kHostThreads];
    try
    {
        for (int w = 1; w < n; ++w)
            t[w] = std::thread(work, w);
    }
    catch (const std::exception &)
    {
    }
    work(0);
    for (auto &x : t)
        if (x.joinable())
            x.join();
}

int host_threads(size_t bytes)
{
    const size_t turns = (bytes + kHostChunk - 1) / kHostChunk;
    return (int)std::max<size_t>(
        1, std::min<size_t>({turns, (size_t)kHostThreads, std::max(1u, std::thread::hardware_concurrency() / 2)}));
}

void host_clear(float *p, size_t count)
{
    const size_t bytes = count * sizeof(float), n = (bytes + kHostChunk - 1) / kHostChunk;
    std::atomic<size_t> next{0};
    on_threads(host_threads(bytes), [&](int) {
        for (size_t i; (i = next++) < n;)
            std::memset(reinterpret_cast<char *>(p) + i * kHostChunk, 0, std::min(kHostChunk, bytes - i * kHostChunk));
    });
}

// The state in host cell order: pulses (ncomp 12, through pv) or stubs (3, at
// soa). Threads take chunks in turn, each through device and pinned memory of
// its own: order on the device, copy out, write to host_out, so that one
// thread's copy runs beside the others' writes. 157^3 cells with stubs, 232 MB
// into fresh memory: 26 ms from pageable copies in one thread, 8.1 here; 64^3, 16 MB: 1.02 and
// 0.87. A state of one chunk goes straight to host_out in one copy: making and
// giving back pinned memory takes longer (24^3, 0.8 MB: 88 us, 152 through
// pinned memory; 32^3, 2 MB: 154 and 214).
int read_back(tlm_ctx *c, float *host_out, const tlm::PulseView *pv, float *soa, int ncomp)
{
    const long long ncell = (long long)c->nx * c->ny * c->nz;
    const long long per = (long long)(kHostChunk / sizeof(float)) / ncomp, nchunk = (ncell + per - 1) / per;
    const int n = host_threads((size_t)ncell * ncomp * sizeof(float));
    const size_t slot = (size_t)std::min(per, ncell) * ncomp;
    float *stage = nullptr, *pin = nullptr;
    int rc = dalloc(c, &stage, slot * n);
    if (rc)
        return rc;
    // cells [c0, c0 + cnt) ordered at d and copied to h
    auto queue = [&](long long c0, long long cnt, float *d, float *h) {
        const unsigned g = (unsigned)((cnt + 255) / 256);
        if (pv)
            hipLaunchKernelGGL(tlm::k_pulses_out, dim3(g), dim3(256), 0, c->stream, *pv, d, c->nxy, c0, cnt);
        else
            hipLaunchKernelGGL(tlm::k_stubs_out, dim3(g), dim3(256), 0, c->stream, soa, d, c->nxy, c->Pp, c0, cnt);
        const hipError_t r = hipGetLastError();
        return r != hipSuccess ? r
                               : hipMemcpyAsync(h, d, (size_t)cnt * ncomp * sizeof(float), hipMemcpyDeviceToHost,
                                                c->stream);
    };
    if (nchunk == 1)
    {
        const hipError_t r = queue(0, ncell, stage, host_out), w = hipStreamSynchronize(c->stream);
        dfree(c, stage);
        return r == hipSuccess && w == hipSuccess ? (int)TLM_OK
                                                  : hip_fail(c, r != hipSuccess ? r : w, "tlm_read_state");
    }
    if (hipHostMalloc((void **)&pin, slot * n * sizeof(float), hipHostMallocDefault) != hipSuccess)
    {
        (void)hipGetLastError(); // without pinned memory straight to host_out
        pin = nullptr;
    }
    hipError_t e = hipSuccess;
    hipEvent_t ev[kHostThreads] = {};
    for (int w = 0; w < n && e == hipSuccess; ++w)
        e = hipEventCreateWithFlags(&ev[w], hipEventDisableTiming);
    std::atomic<long long> next{0};
    std::atomic<int> bad{(int)e};
    if (e == hipSuccess)
        on_threads(n, [&](int w) {
            hipError_t r = hipSetDevice(c->dev);
            for (long long i; r == hipSuccess && bad == hipSuccess && (i = next++) < nchunk;)
            {
                const long long c0 = i * per, cnt = std::min(per, ncell - c0);
                float *h = pin ? pin + slot * w : host_out + c0 * ncomp;
                if ((r = queue(c0, cnt, stage + slot * w, h)) == hipSuccess &&
                    (r = hipEventRecord(ev[w], c->stream)) == hipSuccess &&
                    (r = hipEventSynchronize(ev[w])) == hipSuccess && pin)
                    std::memcpy(host_out + c0 * ncomp, h, (size_t)cnt * ncomp * sizeof(float));
            }
            if (r != hipSuccess)
                bad = (int)r;
        });
    (void)hipStreamSynchronize(c->stream); // before the buffers go, also after a failure
    for (hipEvent_t x : ev)
        if (x)
            (void)hipEventDestroy(x);
    if (pin)
        (void)hipHostFree(pin);
    dfree(c, stage);
    return bad == hipSuccess ? (int)TLM_OK : hip_fail(c, (hipError_t)bad.load(), "tlm_read_state");
}

// Chunked conversion from host cell order to the device layout through a
// bounded staging buffer: pulses (ncomp 12, any storage format, through pv) or
// FP32 stubs (ncomp 3, 64-cell stub blocks at soa).
int convert(tlm_ctx *c, const float *host_in, const tlm::PulseView *pv, float *soa, int ncomp)
{
    const long long ncell = (long long)c->nx * c->ny * c->nz;
    const long long chunk = std::min<long long>(ncell, (long long)8 << 20); // 8 M cells
    float *stage = nullptr;
    int rc = dalloc(c, &stage, (size_t)chunk * ncomp);
    if (rc)
        return rc;
    for (long long c0 = 0; c0 < ncell; c0 += chunk)
    {
        long long cnt = std::min(chunk, ncell - c0);
        int b = 256;
        long long g = (cnt + b - 1) / b;
        hipError_t e = hipMemcpyAsync(stage, host_in + c0 * ncomp, cnt * ncomp * sizeof(float),
                                      hipMemcpyHostToDevice, c->stream);
        if (e != hipSuccess)
        {
            dfree(c, stage);
            return hip_fail(c, e, "hipMemcpyAsync");
        }
        if (pv)
            hipLaunchKernelGGL(tlm::k_pulses_in, dim3((unsigned)g), dim3(b), 0, c->stream, stage,
                               *pv, c->nxy, c0, cnt);
        else
            hipLaunchKernelGGL(tlm::k_stubs_in, dim3((unsigned)g), dim3(b), 0, c->stream, stage,
                               soa, c->nxy, c->Pp, c0, cnt);
        e = hipStreamSynchronize(c->stream);
        if (e != hipSuccess)
        {
            dfree(c, stage);
            return hip_fail(c, e, "hipStreamSynchronize");
        }
    }
    dfree(c, stage);
    return TLM_OK;
}

// 16-bit formats, first run after tlm_upload: decide which slabs keep FP32
// (within `halo` slabs of a soft source), lay the slabs out, choose the
// first scales from the uploaded state and the first injection
// (E_k = exponent of max|state in slab k| + Q_k*|sv(step0)|), and store the
// state rounded to those scales.
int materialize(tlm_ctx *c, int step0)
{
    const int nz = c->nz;
    const long long slab = c->nxy;
    std::vector<float> Q(nz, 0.0f);
    std::vector<char> hot(nz, 0);
    int klo = nz, khi = -1;
    for (size_t s = 0; s < c->src_cells.size(); ++s)
    {
        const int k = (int)(c->src_cells[s] / slab);
        Q[k] = Q[k] + 0.5f * std::fabs(c->src_amp[s]); // list order, as the oracle adds them
        klo = std::min(klo, k);
        khi = std::max(khi, k);
    }
    // one band of FP32 slabs: halo below the lowest source slab to halo above
    // the highest, so the step computes slab offsets without a table lookup
    c->h0 = c->h1 = 0;
    if (c->halo >= 0 && khi >= 0)
    {
        c->h0 = std::max(0, klo - c->halo);
        c->h1 = std::min(nz - 1, khi + c->halo) + 1;
        for (int k = c->h0; k < c->h1; ++k)
            hot[k] = 1;
    }
    std::vector<uint2> sl(nz);
    c->nhot = 0;
    for (int k = 0; k < nz; ++k)
    {
        // 64-cell blocks of 6 pairs: 24 bytes per cell in a 16-bit slab, 48 in an FP32 one
        sl[k] = make_uint2(0u, hot[k] ? 0u : 1u);
        c->nhot += hot[k];
    }
    if ((unsigned long long)c->Pp * 48ULL > (1ULL << 32) - (1ULL << 20))
        return fail(c, TLM_ERR_UNSUPPORTED, "16-bit storage: a slab exceeds 32-bit byte offsets");
    c->PB = (long long)tlm::slab16_base(c->Pp, nz, c->h0, c->h1); // bytes of one buffer
    // slab maxima of the uploaded state
    std::vector<float> M(nz, 0.0f);
    if (!c->pendV.empty())
        for (int k = 0; k < nz; ++k)
        {
            float m = 0.0f;
            const float *v = c->pendV.data() + (size_t)k * slab * 12;
            for (long long i = 0; i < slab * 12; ++i)
                m = std::max(m, std::fabs(v[i]));
            if (!c->pendVs.empty())
            {
                const float *w = c->pendVs.data() + (size_t)k * slab * 3;
                for (long long i = 0; i < slab * 3; ++i)
                    m = std::max(m, std::fabs(w[i]));
            }
            M[k] = m;
        }
    float sv0 = 0.0f;
    HIPCHK(c, hipMemcpy(&sv0, c->sv + step0, sizeof(float), hipMemcpyDeviceToHost));
    std::vector<float> sc(nz), isc(nz);
    for (int k = 0; k < nz; ++k)
    {
        const int E = tlm::plan_exponent(M[k] + Q[k] * std::fabs(sv0));
        sc[k] = tlm::pow2_float(E);
        isc[k] = tlm::pow2_float(-E);
    }
    for (char **buf : {&c->A, &c->B})
    {
        dfree(c, *buf);
        int rc = dalloc(c, buf, (size_t)c->PB);
        if (rc)
            return rc;
    }
    int rc;
    if ((rc = upload(c, &c->slab, sl.data(), sl.size())) ||
        (rc = upload(c, &c->scl[0], sc.data(), sc.size())) ||
        (rc = upload(c, &c->iscl[0], isc.data(), isc.size())) ||
        (rc = upload(c, &c->scl[1], sc.data(), sc.size())) ||
        (rc = upload(c, &c->iscl[1], isc.data(), isc.size())) ||
        (rc = upload(c, &c->mreg, M.data(), M.size())) ||
        (rc = upload(c, &c->qinj, Q.data(), Q.size())) ||
        (rc = upload<float>(c, &c->mpart, nullptr, (size_t)c->strips * nz)) ||
        (rc = upload<int>(c, &c->flag, nullptr, 1)))
        return rc;
    HIPCHK(c, hipMemsetAsync(c->flag, 0, sizeof(int), c->stream));
    HIPCHK(c, hipMemsetAsync(c->A, 0, (size_t)c->PB, c->stream));
    HIPCHK(c, hipMemsetAsync(c->B, 0, (size_t)c->PB, c->stream));
    c->base = step0;
    c->materialized = true;
    if (!c->pendV.empty())
    {
        const tlm::PulseView pv = pulse_view(c, step0);
        if ((rc = convert(c, c->pendV.data(), &pv, nullptr, 12)))
            return rc;
    }
    HIPCHK(c, hipStreamSynchronize(c->stream));
    c->pendV.clear();
    c->pendV.shrink_to_fit();
    c->pendVs.clear();
    c->pendVs.shrink_to_fit();
    return TLM_OK;
}

} // namespace tlmi

using namespace tlmi;

// Cells of a map whose largest id tlm_upload finds on the host.
static constexpr long long kMapHost = 1 << 18;
static uint8_t host_max(const uint8_t *p, size_t n)
{
    uint8_t m = 0;
    for (size_t i = 0; i < n; ++i)
        m = std::max(m, p[i]);
    return m;
}

extern "C" {

int tlm_device_count(void)
{
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess)
        return 0;
    return n;
}

const char *tlm_device_name(int device)
{
    static thread_local char name[256];
    hipDeviceProp_t p;
    if (hipGetDeviceProperties(&p, device) != hipSuccess)
        return "unknown adapter";
    std::snprintf(name, sizeof(name), "%s (%s, %d CUs)", p.name[0] ? p.name : "AMD GPU",
                  p.gcnArchName, p.multiProcessorCount);
    return name;
}

int tlm_create(const tlm_grid_desc *d, tlm_ctx **out)
{
    if (!out)
        return fail(nullptr, TLM_ERR_ARG, "tlm_create: out is NULL");
    *out = nullptr;
    if (!d)
        return fail(nullptr, TLM_ERR_ARG, "tlm_create: desc is NULL");
    if (d->nx <= 0 || d->ny <= 0 || d->nz <= 0)
        return fail(nullptr, TLM_ERR_ARG, "empty grid");
    if (d->pulse_type != TLM_PULSE_F32 && d->pulse_type != TLM_PULSE_F16 &&
        d->pulse_type != TLM_PULSE_BF16)
        return fail(nullptr, TLM_ERR_ARG, "unknown pulse storage type");
    {
        // one pulse plane must be addressable with 32-bit byte offsets
        const long long pp = ((long long)d->nx * d->ny + 63) / 64 * 64;
        if (pp * (long long)d->nz * 4 > (1LL << 32) - (1LL << 20))
            return fail(nullptr, TLM_ERR_UNSUPPORTED,
                        "grid above ~1.07e9 cells: a pulse plane exceeds 32-bit byte offsets");
        // the FP32 step addresses a slab's 12 ports (48 bytes per cell) with
        // 32-bit byte offsets from the slab base
        if (pp * 48 > (1LL << 32) - (1LL << 20))
            return fail(nullptr, TLM_ERR_UNSUPPORTED,
                        "z-slab above ~89e6 cells: its pulses exceed 32-bit byte offsets");
    }
    if (!(d->dl > 0.0f))
        return fail(nullptr, TLM_ERR_ARG, "cell size must be positive");
    int ndev = tlm_device_count();
    if (ndev <= 0)
        return fail(nullptr, TLM_ERR_NO_DEVICE, "no HIP device available");
    if (d->device < 0 || d->device >= ndev)
        return fail(nullptr, TLM_ERR_ARG, "device ordinal out of range");

    tlm_ctx *c = new tlm_ctx;
    c->dev = d->device;
    c->nx = d->nx;
    c->ny = d->ny;
    c->nz = d->nz;
    c->nxy = (long long)c->nx * c->ny;
    c->Pp = (c->nxy + tlm::kWave - 1) / tlm::kWave * tlm::kWave;
    c->P = c->Pp * c->nz;
    c->dl = d->dl;
    c->rho = d->rho;
    c->pf = d->pulse_type;
    // 16-bit pair planes: slabs per wave task, measured (ms a launch at 3 / 4
    // slabs): 64-box scenes 512^3 1.591 / 1.606, 384^3 0.681 / 0.687, 320^3
    // 0.350 / 0.342, 8-box 256^3 0.193 / 0.183
    if (c->pf != TLM_PULSE_F32)
        c->tune.planes = (long long)c->nx * c->ny * c->nz >= (48LL << 20) ? 3 : 4;
    c->halo = d->fp32_halo < 0 ? -1 : (d->fp32_halo == 0 ? 8 : d->fp32_halo);
    c->PB = c->P * 4;
    c->inv_dl = -1.0f / d->dl;
    choose_shape(c);
    auto bail = [&](int rc) {
        g_create_error = c->err;
        tlm_destroy(c);
        return rc;
    };
    hipError_t e = hipSetDevice(c->dev);
    if (e != hipSuccess)
        return bail(hip_fail(c, e, "hipSetDevice"));
    if ((e = hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking)) != hipSuccess)
        return bail(hip_fail(c, e, "hipStreamCreate"));
    for (hipEvent_t *ev : {&c->ev0, &c->ev1, &c->evk0, &c->evk1})
        if ((e = hipEventCreate(ev)) != hipSuccess)
            return bail(hip_fail(c, e, "hipEventCreate"));
    int rc;
    choose_pair(c);
    if (c->pf == TLM_PULSE_F32 &&
        ((rc = dalloc(c, &c->A, (size_t)c->PB * 12)) || (rc = dalloc(c, &c->B, (size_t)c->PB * 12))))
        return bail(rc);
    if ((rc = dalloc(c, &c->code, (size_t)c->P)) || (rc = dalloc(c, &c->epart, energy_parts(c))) ||
        (rc = dalloc(c, &c->epart2, 1024)))
        return bail(rc);
    *out = c;
    return TLM_OK;
}

void tlm_destroy(tlm_ctx *c)
{
    if (!c)
        return;
    if (c->batch)
        (void)tlm_batch_remove(c->batch, c);
    (void)hipSetDevice(c->dev);
    if (c->stream)
        (void)hipStreamSynchronize(c->stream);
    for (void *p : c->owned)
        (void)hipFree(p);
    c->owned.clear();
    for (hipEvent_t ev : {c->ev0, c->ev1, c->evk0, c->evk1})
        if (ev)
            (void)hipEventDestroy(ev);
    for (hipEvent_t ev : c->kev)
        (void)hipEventDestroy(ev);
    if (c->stream)
        (void)hipStreamDestroy(c->stream);
    delete c;
}

const char *tlm_last_error(const tlm_ctx *c)
{
    return c ? c->err.c_str() : g_create_error.c_str();
}

int tlm_upload(tlm_ctx *c, const uint8_t *mat, const float *yhat, const float *ghat, int nmat,
               const float *V, const float *Vs)
{
    if (c && c->batch)
        return fail(c, TLM_ERR_STATE, "context is a batch member");
    if (!c || !mat || nmat < 0 || (nmat > 0 && (!yhat || !ghat)))
        return fail(c, TLM_ERR_ARG, "tlm_upload: bad arguments");
    HIPCHK(c, hipSetDevice(c->dev));
    const long long ncell = (long long)c->nx * c->ny * c->nz;
    // The codes and flags are made on the device, as tlm_upload_mat makes them
    // (of 157^3 cells 8.1 ms in a pass over the host's cells, 0.3 with the
    // map's copy). The map passes through a pulse plane that holds nothing
    // yet, if there is none through memory of its own.
    uint8_t *map = reinterpret_cast<uint8_t *>(c->B), *own = nullptr;
    int rc = TLM_OK, max_id = -1;
    if (c->uploaded || !map)
    {
        if ((rc = dalloc(c, &own, (size_t)ncell)) == TLM_OK)
            map = own;
        else if (!map)
            return rc;
        else
            (void)hipGetLastError(); // the plane that the next step writes: nothing else reads it
    }
    const hipError_t e = hipMemcpyAsync(map, mat, (size_t)ncell, hipMemcpyHostToDevice, c->stream);
    rc = e == hipSuccess ? (int)TLM_OK : hip_fail(c, e, "hipMemcpyAsync");
    // the largest id, of a small map sooner on the host than by a launch and a
    // wait for its result (first upload of a context 4^3 70 us, 96 on the device,
    // 24^3 73 and 100, 64^3 134 and 157; 80^3 on the device 190)
    if (ncell <= kMapHost)
        max_id = (int)std::max<unsigned>(1u, host_max(mat, (size_t)ncell)) - 2;
    else if (!rc)
        rc = largest_id(c, map, &max_id);
    if (!rc)
        rc = build_codes(c, map, nmat, max_id);
    (void)hipStreamSynchronize(c->stream); // before the map goes, also after a failure
    dfree(c, own);
    return rc ? rc : install_material(c, max_id >= 0, yhat, ghat, nmat, V, Vs);
}

} // extern "C"

namespace tlmi {

int install_material(tlm_ctx *c, bool any_diel, const float *yhat, const float *ghat, int nmat,
                     const float *V, const float *Vs)
{
    const long long ncell = (long long)c->nx * c->ny * c->nz;
    // per-material (yh, gh, den), den = 4 + yh + gh as in TlmSolver.cpp:90
    std::vector<float4> props(std::max(1, nmat));
    for (int i = 0; i < nmat; ++i)
    {
        float den = 4.0f + yhat[i] + ghat[i];
        props[i] = make_float4(yhat[i], ghat[i], den, 0.f);
    }
    int rc = upload(c, &c->props, props.data(), props.size());
    if (rc)
        return rc;
    c->nmat = nmat;
    if (c->pf == TLM_PULSE_F32)
    {
        HIPCHK(c, hipMemsetAsync(c->A, 0, (size_t)c->PB * 12, c->stream));
        HIPCHK(c, hipMemsetAsync(c->B, 0, (size_t)c->PB * 12, c->stream));
    }
    c->stubs = false;
    dfree(c, c->Vs);
    c->pair_ready = c->pair_refused = false;
    if (any_diel)
    {
        if ((rc = dalloc(c, &c->Vs, (size_t)c->P * 3)))
            return rc;
        c->stubs = true;
        HIPCHK(c, hipMemsetAsync(c->Vs, 0, (size_t)c->P * 3 * sizeof(float), c->stream));
    }
    else
        dfree(c, c->Vs2);
    HIPCHK(c, hipStreamSynchronize(c->stream));
    if (c->pf == TLM_PULSE_F32)
    {
        const tlm::PulseView pv = pulse_view(c, 0);
        if (V && (rc = convert(c, V, &pv, nullptr, 12)))
            return rc;
    }
    else
    {
        // the 16-bit scales depend on the sources and the first step: the
        // state is stored at the first tlm_run
        c->materialized = false;
        c->pendV.clear();
        c->pendVs.clear();
        if (V)
        {
            c->pendV.assign(V, V + (size_t)ncell * 12);
            if (Vs && c->stubs)
                c->pendVs.assign(Vs, Vs + (size_t)ncell * 3);
        }
    }
    if (Vs && c->stubs && (rc = convert(c, Vs, nullptr, c->Vs, 3)))
        return rc;
    c->uploaded = true;
    c->launches = c->pairs = 0;
    c->energy_steps.clear();
    c->steps_run_hi = 0;
    c->dft_done = 0;
    return TLM_OK;
}

} // namespace tlmi

extern "C" {

int tlm_set_sources(tlm_ctx *c, const int64_t *cells, const int32_t *pol, const float *amp, int n)
{
    if (c && c->batch)
        return fail(c, TLM_ERR_STATE, "context is a batch member");
    if (!c || n < 0 || (n > 0 && (!cells || !pol || !amp)))
        return fail(c, TLM_ERR_ARG, "tlm_set_sources: bad arguments");
    if (c->pf != TLM_PULSE_F32 && c->materialized)
        return fail(c, TLM_ERR_STATE,
                    "16-bit pulse storage: sources are fixed once the first step has run");
    // group by cell, keeping list order within a cell
    std::map<long long, std::vector<int>> by;
    for (int s = 0; s < n; ++s)
    {
        if (!cell_ok(c, cells[s]) || pol[s] < 0 || pol[s] > 2)
            return fail(c, TLM_ERR_ARG, "source cell or polarisation out of range");
        by[cells[s]].push_back(s);
    }
    std::vector<long long> uc;
    std::vector<int> ub, sp;
    std::vector<float> sa;
    for (auto &kv : by)
    {
        uc.push_back(padded_cell(c, kv.first));
        ub.push_back((int)sp.size());
        for (int s : kv.second)
        {
            sp.push_back(pol[s]);
            sa.push_back(amp[s]);
        }
    }
    ub.push_back((int)sp.size());
    c->src_cells.assign(cells, cells + n);
    c->src_amp.assign(amp, amp + n);
    int rc;
    if ((rc = upload(c, &c->ucell, uc.data(), uc.size())) ||
        (rc = upload(c, &c->ubeg, ub.data(), ub.size())) ||
        (rc = upload(c, &c->spol, sp.data(), sp.size())) ||
        (rc = upload(c, &c->samp, sa.data(), sa.size())))
        return rc;
    c->nuniq = (int)uc.size();
    c->fold_marked = false;
    return TLM_OK;
}

int tlm_set_schedule(tlm_ctx *c, const float *sv, const float *cph, const float *sph, int nsteps,
                     int settle)
{
    if (c && c->batch)
        return fail(c, TLM_ERR_STATE, "context is a batch member");
    if (!c || nsteps <= 0 || !sv || !cph || !sph)
        return fail(c, TLM_ERR_ARG, "tlm_set_schedule: bad arguments");
    int rc;
    if ((rc = upload(c, &c->sv, sv, nsteps)) || (rc = upload(c, &c->cph, cph, nsteps)) ||
        (rc = upload(c, &c->sph, sph, nsteps)))
        return rc;
    c->sv_host.assign(sv, sv + nsteps);
    c->nsteps = nsteps;
    c->settle = settle;
    c->nfreq = 0; // DFT tables are sized by the schedule: set them again
    c->dft_done = 0;
    const int ne = c->every > 0 ? nsteps / c->every + 1 : 1;
    dfree(c, c->energy);
    if ((rc = dalloc(c, &c->energy, ne)))
        return rc;
    c->energy_steps.clear();
    // record buffers that scale with the schedule length
    if (c->np > 0)
    {
        dfree(c, c->prec);
        if ((rc = dalloc(c, &c->prec, (size_t)nsteps * c->np * 2)))
            return rc;
        HIPCHK(c, hipMemset(c->prec, 0, (size_t)nsteps * c->np * 2 * sizeof(float)));
    }
    if (c->npr > 0)
    {
        dfree(c, c->prrec);
        if ((rc = dalloc(c, &c->prrec, (size_t)nsteps * c->npr * 3)))
            return rc;
        HIPCHK(c, hipMemset(c->prrec, 0, (size_t)nsteps * c->npr * 3 * sizeof(float)));
    }
    return TLM_OK;
}

int tlm_set_energy_every(tlm_ctx *c, int every)
{
    if (!c || every < 0)
        return fail(c, TLM_ERR_ARG, "tlm_set_energy_every: bad arguments");
    c->every = every;
    if (c->nsteps > 0)
    {
        dfree(c, c->energy);
        int rc = dalloc(c, &c->energy, every > 0 ? c->nsteps / every + 1 : 1);
        if (rc)
            return rc;
    }
    c->energy_steps.clear();
    return TLM_OK;
}

int tlm_set_plane(tlm_ctx *c, int axis, int index)
{
    if (c && c->batch)
        return fail(c, TLM_ERR_STATE, "context is a batch member");
    if (!c || axis > 2)
        return fail(c, TLM_ERR_ARG, "tlm_set_plane: bad arguments");
    dfree(c, c->plane);
    c->pa = axis < 0 ? -1 : axis;
    c->plane_step = -1;
    if (c->pa < 0)
        return TLM_OK;
    const int nn[3] = {c->nx, c->ny, c->nz};
    const int a1 = (axis == 0) ? 1 : 0, a2 = (axis == 2) ? 1 : 2;
    c->pn1 = nn[a1];
    c->pn2 = nn[a2];
    c->pidx = std::min(std::max(index, 0), nn[axis] - 1);
    int rc = dalloc(c, &c->plane, (size_t)c->pn1 * c->pn2);
    if (rc)
        return rc;
    HIPCHK(c, hipMemset(c->plane, 0, (size_t)c->pn1 * c->pn2 * sizeof(float)));
    return TLM_OK;
}

int tlm_set_frames(tlm_ctx *c, int every, int max_frames)
{
    if (c && c->batch)
        return fail(c, TLM_ERR_STATE, "context is a batch member");
    if (!c || every < 0 || max_frames < 0)
        return fail(c, TLM_ERR_ARG, "tlm_set_frames: bad arguments");
    dfree(c, c->frame_js);
    dfree(c, c->frame_plane);
    c->frame_steps.clear();
    c->frame_plane_step.clear();
    c->frame_every = (max_frames > 0) ? every : 0;
    c->frame_max = max_frames;
    if (c->frame_every == 0)
        return TLM_OK;
    int rc;
    if ((rc = dalloc(c, &c->frame_js, (size_t)max_frames * std::max(1, c->nf))))
        return rc;
    if (c->pa >= 0 &&
        (rc = dalloc(c, &c->frame_plane, (size_t)max_frames * c->pn1 * c->pn2)))
        return rc;
    return TLM_OK;
}

int tlm_read_plane(tlm_ctx *c, float *out, int *n1, int *n2, int *step)
{
    if (!c)
        return TLM_ERR_ARG;
    if (n1)
        *n1 = c->pa >= 0 ? c->pn1 : 0;
    if (n2)
        *n2 = c->pa >= 0 ? c->pn2 : 0;
    if (step)
        *step = c->pa >= 0 ? c->plane_step : -1;
    if (out && c->pa >= 0)
    {
        HIPCHK(c, hipStreamSynchronize(c->stream));
        HIPCHK(c, hipMemcpy(out, c->plane, (size_t)c->pn1 * c->pn2 * sizeof(float),
                            hipMemcpyDeviceToHost));
    }
    return TLM_OK;
}

int tlm_read_frames(tlm_ctx *c, int32_t *steps, float *js, float *planes, int cap)
{
    if (!c || cap < 0)
        return fail(c, TLM_ERR_ARG, "tlm_read_frames: bad arguments");
    const int cnt = (int)c->frame_steps.size();
    const int m = std::min(cap, cnt);
    if (m > 0)
    {
        HIPCHK(c, hipStreamSynchronize(c->stream));
        if (steps)
            for (int f = 0; f < m; ++f)
                steps[f] = c->frame_steps[f];
        if (js && c->nf > 0)
            HIPCHK(c, hipMemcpy(js, c->frame_js, (size_t)m * c->nf * sizeof(float),
                                hipMemcpyDeviceToHost));
        if (planes && c->pa >= 0 && c->frame_plane)
            HIPCHK(c, hipMemcpy(planes, c->frame_plane, (size_t)m * c->pn1 * c->pn2 * sizeof(float),
                                hipMemcpyDeviceToHost));
    }
    return cnt;
}

int tlm_set_probes(tlm_ctx *c, const int64_t *cells, int n, float inv_dl)
{
    if (c && c->batch)
        return fail(c, TLM_ERR_STATE, "context is a batch member");
    if (!c || n < 0 || (n > 0 && !cells))
        return fail(c, TLM_ERR_ARG, "tlm_set_probes: bad arguments");
    if (c->nsteps <= 0)
        return fail(c, TLM_ERR_STATE, "tlm_set_probes before tlm_set_schedule");
    std::vector<long long> pc(n);
    for (int i = 0; i < n; ++i)
    {
        if (!cell_ok(c, cells[i]))
            return fail(c, TLM_ERR_ARG, "probe cell out of range");
        pc[i] = padded_cell(c, cells[i]);
    }
    int rc;
    if ((rc = upload(c, &c->prcell, pc.data(), pc.size())))
        return rc;
    c->npr = n;
    c->inv_dl = inv_dl;
    dfree(c, c->prrec);
    if ((rc = dalloc(c, &c->prrec, (size_t)c->nsteps * std::max(1, n) * 3)))
        return rc;
    HIPCHK(c, hipMemset(c->prrec, 0, (size_t)c->nsteps * std::max(1, n) * 3 * sizeof(float)));
    c->nfreq = 0;
    return TLM_OK;
}

int tlm_set_probe_dft(tlm_ctx *c, const double *ctab, const double *stab, int nfreq)
{
    if (c && c->batch)
        return fail(c, TLM_ERR_STATE, "context is a batch member");
    if (!c || nfreq < 0 || (nfreq > 0 && (!ctab || !stab)))
        return fail(c, TLM_ERR_ARG, "tlm_set_probe_dft: bad arguments");
    if (c->nsteps <= 0)
        return fail(c, TLM_ERR_STATE, "tlm_set_probe_dft before tlm_set_schedule");
    int rc;
    const size_t tab = (size_t)c->nsteps * nfreq;
    if ((rc = upload(c, &c->ctab, ctab, tab)) || (rc = upload(c, &c->stab, stab, tab)))
        return rc;
    const size_t acc = (size_t)std::max(1, c->npr) * 3 * std::max(1, nfreq);
    dfree(c, c->dft_re);
    dfree(c, c->dft_im);
    if ((rc = dalloc(c, &c->dft_re, acc)) || (rc = dalloc(c, &c->dft_im, acc)))
        return rc;
    HIPCHK(c, hipMemset(c->dft_re, 0, acc * sizeof(double)));
    HIPCHK(c, hipMemset(c->dft_im, 0, acc * sizeof(double)));
    c->nfreq = nfreq;
    c->dft_done = 0;
    return TLM_OK;
}

int tlm_set_ports(tlm_ctx *c, const int64_t *cells, const int32_t *off, const int32_t *pol, int np)
{
    if (c && c->batch)
        return fail(c, TLM_ERR_STATE, "context is a batch member");
    if (!c || np < 0 || (np > 0 && (!off || !pol)))
        return fail(c, TLM_ERR_ARG, "tlm_set_ports: bad arguments");
    if (c->nsteps <= 0)
        return fail(c, TLM_ERR_STATE, "tlm_set_ports before tlm_set_schedule");
    std::vector<long long> pc;
    std::vector<long long> loop(4 * (size_t)std::max(1, np), 0);
    std::vector<int> po(np + 1), pp(np);
    const long long stride[3] = {1, c->nx, (long long)c->nx * c->ny};
    for (int p = 0; p < np; ++p)
    {
        if (pol[p] < 0 || pol[p] > 2 || off[p + 1] < off[p])
            return fail(c, TLM_ERR_ARG, "bad port description");
        po[p] = (int)pc.size();
        pp[p] = pol[p];
        for (int s = off[p]; s < off[p + 1]; ++s)
        {
            if (!cell_ok(c, cells[s]))
                return fail(c, TLM_ERR_ARG, "port cell out of range");
            pc.push_back(padded_cell(c, cells[s]));
        }
        const int cnt = off[p + 1] - off[p];
        if (cnt > 0)
        {
            // Ampere loop neighbours by linear index, as TlmSolver.cpp:687-698
            long long mid = cells[off[p] + cnt / 2];
            int t1 = (pol[p] + 1) % 3, t2 = (pol[p] + 2) % 3;
            long long nb[4] = {mid + stride[t1], mid - stride[t1], mid + stride[t2], mid - stride[t2]};
            for (int q = 0; q < 4; ++q)
            {
                if (!cell_ok(c, nb[q]))
                    return fail(c, TLM_ERR_ARG, "port current loop leaves the grid");
                loop[4 * p + q] = padded_cell(c, nb[q]);
            }
        }
    }
    po[np] = (int)pc.size();
    int rc;
    if ((rc = upload(c, &c->pcells, pc.data(), pc.size())) ||
        (rc = upload(c, &c->poff, po.data(), po.size())) ||
        (rc = upload(c, &c->ppol, pp.data(), pp.size())) ||
        (rc = upload(c, &c->ploop, loop.data(), loop.size())))
        return rc;
    c->np = np;
    dfree(c, c->prec);
    if ((rc = dalloc(c, &c->prec, (size_t)c->nsteps * std::max(1, np) * 2)))
        return rc;
    HIPCHK(c, hipMemset(c->prec, 0, (size_t)c->nsteps * std::max(1, np) * 2 * sizeof(float)));
    return TLM_OK;
}

int tlm_set_faces(tlm_ctx *c, const int64_t *cells, const int32_t *axes, int n)
{
    if (c && c->batch)
        return fail(c, TLM_ERR_STATE, "context is a batch member");
    if (!c || n < 0 || (n > 0 && (!cells || !axes)))
        return fail(c, TLM_ERR_ARG, "tlm_set_faces: bad arguments");
    std::vector<long long> fc(n);
    std::vector<int> fa(n);
    for (int i = 0; i < n; ++i)
    {
        if (!cell_ok(c, cells[i]) || axes[i] < 0 || axes[i] > 2)
            return fail(c, TLM_ERR_ARG, "face cell or axis out of range");
        fc[i] = padded_cell(c, cells[i]);
        fa[i] = axes[i];
    }
    int rc;
    if ((rc = upload(c, &c->fcell, fc.data(), fc.size())) ||
        (rc = upload(c, &c->faxis, fa.data(), fa.size())))
        return rc;
    dfree(c, c->js_inst);
    dfree(c, c->js_dft4);
    if ((rc = dalloc(c, &c->js_inst, std::max(1, n))) ||
        (rc = dalloc(c, &c->js_dft4, 4 * (size_t)std::max(1, n))))
        return rc;
    HIPCHK(c, hipMemset(c->js_inst, 0, std::max(1, n) * sizeof(float)));
    HIPCHK(c, hipMemset(c->js_dft4, 0, 4 * (size_t)std::max(1, n) * sizeof(float)));
    c->nf = n;
    return TLM_OK;
}

int tlm_set_huygens(tlm_ctx *c, const int64_t *cells, const int32_t *axes, int n)
{
    if (c && c->batch)
        return fail(c, TLM_ERR_STATE, "context is a batch member");
    if (!c || n < 0 || (n > 0 && (!cells || !axes)))
        return fail(c, TLM_ERR_ARG, "tlm_set_huygens: bad arguments");
    std::vector<long long> hc(n);
    std::vector<int> ha(n);
    for (int i = 0; i < n; ++i)
    {
        if (!cell_ok(c, cells[i]) || axes[i] < 0 || axes[i] > 2)
            return fail(c, TLM_ERR_ARG, "Huygens cell or axis out of range");
        hc[i] = padded_cell(c, cells[i]);
        ha[i] = axes[i];
    }
    int rc;
    c->hlat = HuyLattice{};
    c->hlat_known = false;
    if ((rc = upload(c, &c->hcell, hc.data(), hc.size())) ||
        (rc = upload(c, &c->haxis, ha.data(), ha.size())))
        return rc;
    dfree(c, c->huy8);
    if ((rc = dalloc(c, &c->huy8, 8 * (size_t)std::max(1, n))))
        return rc;
    HIPCHK(c, hipMemset(c->huy8, 0, 8 * (size_t)std::max(1, n) * sizeof(float)));
    c->nh = n;
    return TLM_OK;
}

int tlm_run(tlm_ctx *c, int step0, int nsteps)
{
    if (!c)
        return TLM_ERR_ARG;
    return queue_steps(c, step0, nsteps, 0, nullptr, nullptr);
}

int tlm_sync(tlm_ctx *c)
{
    if (!c)
        return TLM_ERR_ARG;
    HIPCHK(c, hipSetDevice(c->dev));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    HIPCHK(c, hipGetLastError());
    if (c->flag)
    {
        int f = 0;
        HIPCHK(c, hipMemcpy(&f, c->flag, sizeof(int), hipMemcpyDeviceToHost));
        if (f)
            return fail(c, TLM_ERR_RANGE,
                        "16-bit pulse storage: a value exceeded the range its slab scale allows");
    }
    return TLM_OK;
}

int tlm_read_scales(tlm_ctx *c, float *scale, float *smax, int32_t *fmt)
{
    if (!c)
        return TLM_ERR_ARG;
    if (c->pf == TLM_PULSE_F32 || !c->materialized)
        return 0;
    HIPCHK(c, hipSetDevice(c->dev));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    if (scale)
        HIPCHK(c, hipMemcpy(scale, c->scl[scale_buf(c, c->next_step)], c->nz * sizeof(float),
                            hipMemcpyDeviceToHost));
    if (smax)
        HIPCHK(c, hipMemcpy(smax, c->mreg, c->nz * sizeof(float), hipMemcpyDeviceToHost));
    if (fmt)
    {
        std::vector<uint2> sl(c->nz);
        HIPCHK(c, hipMemcpy(sl.data(), c->slab, c->nz * sizeof(uint2), hipMemcpyDeviceToHost));
        for (int k = 0; k < c->nz; ++k)
            fmt[k] = sl[k].y ? c->pf : TLM_PULSE_F32;
    }
    return c->nz;
}

int tlm_device_memory(int device, size_t *free_bytes, size_t *total_bytes)
{
    if (device < 0 || device >= tlm_device_count())
        return TLM_ERR_NO_DEVICE;
    if (hipSetDevice(device) != hipSuccess)
        return TLM_ERR_HIP;
    size_t f = 0, t = 0;
    if (hipMemGetInfo(&f, &t) != hipSuccess)
        return TLM_ERR_HIP;
    if (free_bytes)
        *free_bytes = f;
    if (total_bytes)
        *total_bytes = t;
    return TLM_OK;
}

int64_t tlm_estimate_bytes(const tlm_grid_desc *d, int has_stubs)
{
    if (!d || d->nx <= 0 || d->ny <= 0 || d->nz <= 0)
        return TLM_ERR_ARG;
    const long long Pp = ((long long)d->nx * d->ny + 63) / 64 * 64, P = Pp * d->nz;
    const long long sp = d->pulse_type == TLM_PULSE_F32 ? 4 : 2; // FP32 halo slabs not counted
    long long bytes = 2 * 12 * P * sp + 2 * P;                   // pulses A, B and cell codes
    if (has_stubs)
        bytes += 3 * P * 4;
    bytes += (P / 64) * 8 + (1 << 20); // energy / slab-maximum partials, small tables
    return bytes;
}

int tlm_device_encode(int device, int fmt, const float *in, float inv_scale, uint16_t *out,
                      int64_t n)
{
    if ((fmt != TLM_PULSE_F16 && fmt != TLM_PULSE_BF16) || n < 0 || (n && (!in || !out)))
        return TLM_ERR_ARG;
    if (device < 0 || device >= tlm_device_count())
        return TLM_ERR_NO_DEVICE;
    if (hipSetDevice(device) != hipSuccess)
        return TLM_ERR_HIP;
    if (n == 0)
        return TLM_OK;
    float *din = nullptr;
    unsigned short *dout = nullptr;
    if (hipMalloc((void **)&din, n * sizeof(float)) != hipSuccess)
        return TLM_ERR_NOMEM;
    if (hipMalloc((void **)&dout, n * sizeof(unsigned short)) != hipSuccess)
    {
        (void)hipFree(din);
        return TLM_ERR_NOMEM;
    }
    int rc = TLM_OK;
    if (hipMemcpy(din, in, n * sizeof(float), hipMemcpyHostToDevice) != hipSuccess)
        rc = TLM_ERR_HIP;
    else
    {
        const int b = 256;
        hipLaunchKernelGGL(tlm::k_encode, dim3((unsigned)((n + b - 1) / b)), dim3(b), 0, 0, fmt, din,
                           inv_scale, dout, (long long)n);
        if (hipDeviceSynchronize() != hipSuccess ||
            hipMemcpy(out, dout, n * sizeof(unsigned short), hipMemcpyDeviceToHost) != hipSuccess)
            rc = TLM_ERR_HIP;
    }
    (void)hipFree(din);
    (void)hipFree(dout);
    return rc;
}

int tlm_time_steps(tlm_ctx *c, int step0, int nsteps, int kernel_every, float *ms_total,
                   float *ms_kernel, int *nkernel)
{
    if (!c)
        return TLM_ERR_ARG;
    if (kernel_every < 0)
        return fail(c, TLM_ERR_ARG, "tlm_time_steps: kernel_every < 0");
    if (ms_kernel)
        *ms_kernel = 0.f;
    if (nkernel)
        *nkernel = 0;
    c->timed_launches = c->timed_pairs = 0;
    HIPCHK(c, hipSetDevice(c->dev));
    HIPCHK(c, hipEventRecord(c->ev0, c->stream));
    int rc = queue_steps(c, step0, nsteps, ms_kernel ? kernel_every : 0, ms_kernel, nkernel);
    if (rc)
        return rc;
    HIPCHK(c, hipEventRecord(c->ev1, c->stream));
    HIPCHK(c, hipEventSynchronize(c->ev1));
    float ms = 0.f;
    HIPCHK(c, hipEventElapsedTime(&ms, c->ev0, c->ev1));
    if (ms_total)
        *ms_total = ms;
    return TLM_OK;
}

int tlm_timed_launches(const tlm_ctx *c, int *launches, int *pairs)
{
    if (!c)
        return TLM_ERR_ARG;
    if (launches)
        *launches = c->timed_launches;
    if (pairs)
        *pairs = c->timed_pairs;
    return TLM_OK;
}

int tlm_step_launches(const tlm_ctx *c, int64_t *launches, int64_t *pairs)
{
    if (!c)
        return TLM_ERR_ARG;
    if (launches)
        *launches = c->launches;
    if (pairs)
        *pairs = c->pairs;
    return TLM_OK;
}

int tlm_launch_shape(const tlm_ctx *c, int *rows, int *planes, int *groups, int *threads)
{
    if (!c)
        return TLM_ERR_ARG;
    if (rows)
        *rows = c->strips;
    if (planes)
        *planes = c->zc;
    if (groups)
        *groups = c->blocks;
    if (threads)
        *threads = c->wpb * tlm::kWave;
    return TLM_OK;
}

int tlm_set_tuning(tlm_ctx *c, const tlm_tuning *t)
{
    if (c && c->batch)
        return fail(c, TLM_ERR_STATE, "context is a batch member");
    if (!c || !t || t->kernel != 0 || t->planes < 0 || t->block_waves < 0 ||
        t->block_waves > 4 || t->nontemporal < 0 || t->nontemporal > 2 || t->grid_blocks < 0 ||
        t->fold < 0 || t->fold > 2 || t->occupancy < -1 || (t->occupancy > 0 && t->occupancy < 3) ||
        t->occupancy > 8)
        return fail(c, TLM_ERR_ARG, "tlm_set_tuning: bad arguments");
    HIPCHK(c, hipStreamSynchronize(c->stream));
    c->tune = *t;
    choose_shape(c);
    return TLM_OK;
}

int tlm_get_tuning(const tlm_ctx *c, tlm_tuning *t)
{
    if (!c || !t)
        return TLM_ERR_ARG;
    *t = c->tune;
    return TLM_OK;
}

int tlm_read_state(tlm_ctx *c, float *V, float *Vs)
{
    if (!c || !V)
        return fail(c, TLM_ERR_ARG, "tlm_read_state: bad arguments");
    HIPCHK(c, hipSetDevice(c->dev));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    const size_t ncell = (size_t)c->nx * c->ny * c->nz;
    if (c->pf != TLM_PULSE_F32 && !c->materialized)
    {
        // not run yet: the uploaded state
        if (c->pendV.empty())
            host_clear(V, 12 * ncell);
        else
            std::memcpy(V, c->pendV.data(), sizeof(float) * 12 * ncell);
    }
    else
    {
        const tlm::PulseView pv = pulse_view(c, c->next_step);
        int rc = read_back(c, V, &pv, nullptr, 12);
        if (rc)
            return rc;
    }
    if (Vs)
    {
        if (c->stubs)
            return read_back(c, Vs, nullptr, c->Vs, 3);
        host_clear(Vs, 3 * ncell);
    }
    return TLM_OK;
}

int tlm_read_probes(tlm_ctx *c, int step0, int nsteps, float *e)
{
    if (!c || step0 < 0 || nsteps < 0 || step0 + nsteps > c->nsteps || (!e && nsteps))
        return fail(c, TLM_ERR_ARG, "tlm_read_probes: bad arguments");
    if (c->npr == 0 || nsteps == 0)
        return TLM_OK;
    HIPCHK(c, hipSetDevice(c->dev));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    HIPCHK(c, hipMemcpy(e, c->prrec + (size_t)step0 * c->npr * 3,
                        (size_t)nsteps * c->npr * 3 * sizeof(float), hipMemcpyDeviceToHost));
    return TLM_OK;
}

int tlm_read_probe_dft(tlm_ctx *c, double *re, double *im)
{
    if (!c || !re || !im)
        return fail(c, TLM_ERR_ARG, "tlm_read_probe_dft: bad arguments");
    if (c->npr == 0 || c->nfreq == 0)
        return TLM_OK;
    HIPCHK(c, hipSetDevice(c->dev));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    const size_t n = (size_t)c->npr * 3 * c->nfreq;
    HIPCHK(c, hipMemcpy(re, c->dft_re, n * sizeof(double), hipMemcpyDeviceToHost));
    HIPCHK(c, hipMemcpy(im, c->dft_im, n * sizeof(double), hipMemcpyDeviceToHost));
    return TLM_OK;
}

int tlm_read_ports(tlm_ctx *c, int step0, int nsteps, float *vi)
{
    if (!c || step0 < 0 || nsteps < 0 || step0 + nsteps > c->nsteps || (!vi && nsteps))
        return fail(c, TLM_ERR_ARG, "tlm_read_ports: bad arguments");
    if (c->np == 0 || nsteps == 0)
        return TLM_OK;
    HIPCHK(c, hipSetDevice(c->dev));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    HIPCHK(c, hipMemcpy(vi, c->prec + (size_t)step0 * c->np * 2,
                        (size_t)nsteps * c->np * 2 * sizeof(float), hipMemcpyDeviceToHost));
    return TLM_OK;
}

int tlm_read_js(tlm_ctx *c, float *inst, float *dft4)
{
    if (!c)
        return TLM_ERR_ARG;
    if (c->nf == 0)
        return TLM_OK;
    HIPCHK(c, hipSetDevice(c->dev));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    if (inst)
        HIPCHK(c, hipMemcpy(inst, c->js_inst, (size_t)c->nf * sizeof(float), hipMemcpyDeviceToHost));
    if (dft4)
        HIPCHK(c, hipMemcpy(dft4, c->js_dft4, (size_t)c->nf * 4 * sizeof(float),
                            hipMemcpyDeviceToHost));
    return TLM_OK;
}

int tlm_read_huygens(tlm_ctx *c, float *dft8)
{
    if (!c || !dft8)
        return fail(c, TLM_ERR_ARG, "tlm_read_huygens: bad arguments");
    if (c->nh == 0)
        return TLM_OK;
    HIPCHK(c, hipSetDevice(c->dev));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    HIPCHK(c, hipMemcpy(dft8, c->huy8, (size_t)c->nh * 8 * sizeof(float), hipMemcpyDeviceToHost));
    return TLM_OK;
}

int tlm_read_energy(tlm_ctx *c, int32_t *steps, double *vals, int cap)
{
    if (!c || cap < 0)
        return fail(c, TLM_ERR_ARG, "tlm_read_energy: bad arguments");
    HIPCHK(c, hipSetDevice(c->dev));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    std::vector<int> idx;
    for (size_t i = 0; i < c->energy_steps.size(); ++i)
        if (c->energy_steps[i] >= 0)
            idx.push_back((int)i);
    const int cnt = (int)idx.size();
    if (cap > 0 && (steps || vals))
    {
        std::vector<double> all(c->energy_steps.size());
        if (!all.empty())
            HIPCHK(c, hipMemcpy(all.data(), c->energy, all.size() * sizeof(double),
                                hipMemcpyDeviceToHost));
        for (int q = 0; q < std::min(cap, cnt); ++q)
        {
            if (steps)
                steps[q] = c->energy_steps[idx[q]];
            if (vals)
                vals[q] = all[idx[q]];
        }
    }
    return cnt;
}

int tlm_copy_bandwidth(int device, size_t bytes, int iters, float *gbps, float *ms_per_copy)
{
    if (bytes < 16 || iters <= 0)
        return TLM_ERR_ARG;
    if (tlm_device_count() <= device || device < 0)
        return TLM_ERR_NO_DEVICE;
    if (hipSetDevice(device) != hipSuccess)
        return TLM_ERR_HIP;
    const size_t n4 = bytes / 16;
    float4 *src = nullptr, *dst = nullptr;
    if (hipMalloc((void **)&src, n4 * 16) != hipSuccess)
        return TLM_ERR_NOMEM;
    if (hipMalloc((void **)&dst, n4 * 16) != hipSuccess)
    {
        (void)hipFree(src);
        return TLM_ERR_NOMEM;
    }
    hipEvent_t e0, e1;
    (void)hipEventCreate(&e0);
    (void)hipEventCreate(&e1);
    (void)hipMemset(src, 0, n4 * 16);
    const int b = 256;
    const unsigned g = (unsigned)std::min<size_t>((n4 + b - 1) / b, 1u << 20);
    hipLaunchKernelGGL(tlm::k_copy, dim3(g), dim3(b), 0, 0, src, dst, (long long)n4);
    (void)hipEventRecord(e0, 0);
    for (int i = 0; i < iters; ++i)
        hipLaunchKernelGGL(tlm::k_copy, dim3(g), dim3(b), 0, 0, src, dst, (long long)n4);
    (void)hipEventRecord(e1, 0);
    hipError_t e = hipEventSynchronize(e1);
    float ms = 0.f;
    (void)hipEventElapsedTime(&ms, e0, e1);
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    (void)hipFree(src);
    (void)hipFree(dst);
    if (e != hipSuccess)
        return TLM_ERR_HIP;
    if (ms_per_copy)
        *ms_per_copy = ms / iters;
    if (gbps)
        *gbps = (float)(2.0 * n4 * 16 * iters / (ms * 1e-3) / 1e9);
    return TLM_OK;
}

float tlm_scatter_unitarity_error(float epsr)
{
    if (tlm_device_count() <= 0)
        return (float)TLM_ERR_NO_DEVICE;
    const bool diel = epsr > 1.0f;
    const int NP = diel ? 15 : 12;
    float yh = diel ? 4.0f * (epsr - 1.0f) : 0.0f;
    float den = 4.0f + yh + 0.0f;
    float *dS = nullptr;
    if (hipMalloc((void **)&dS, 15 * 15 * sizeof(float)) != hipSuccess)
        return (float)TLM_ERR_NOMEM;
    hipLaunchKernelGGL(tlm::k_scatter_columns, dim3(1), dim3(64), 0, 0, yh, den, diel ? 1 : 0, dS);
    float S[15 * 15];
    hipError_t e = hipMemcpy(S, dS, sizeof(S), hipMemcpyDeviceToHost);
    (void)hipFree(dS);
    if (e != hipSuccess)
        return (float)TLM_ERR_HIP;
    // S^T W S against W with W = (1 x 12, yh x 3), as TlmSolver.cpp:141-169
    float W[15];
    for (int i = 0; i < 15; ++i)
        W[i] = i < 12 ? 1.0f : yh;
    float maxErr = 0.0f;
    for (int a = 0; a < NP; ++a)
        for (int b = 0; b < NP; ++b)
        {
            float dot = 0.0f;
            for (int r = 0; r < NP; ++r)
                dot += W[r] * S[r * 15 + a] * S[r * 15 + b];
            float want = (a == b) ? W[a] : 0.0f;
            maxErr = std::max(maxErr, std::fabs(dot - want));
        }
    return maxErr;
}

int64_t tlm_build_pec_faces(int nx, int ny, int nz, const uint8_t *mat, int64_t *cells,
                            int32_t *axes, int32_t *signs, int64_t cap)
{
    if (!mat || nx <= 0 || ny <= 0 || nz <= 0)
        return 0;
    const long long dirs[3] = {1, nx, (long long)nx * ny};
    const int nn[3] = {nx, ny, nz};
    int64_t cnt = 0;
    for (int k = 0; k < nz; ++k)
        for (int j = 0; j < ny; ++j)
            for (int i = 0; i < nx; ++i)
            {
                // a row's next PEC cell by memchr (157 x 131 x 143 cells, one plane PEC, twice:
                // 0.4 ms; by a byte at a time 1.8 or 2.4 on one host, as the loop happened to be placed)
                const uint8_t *row = mat + ((long long)k * ny + j) * nx;
                if (row[i] != 1)
                {
                    const void *p = std::memchr(row + i, 1, (size_t)(nx - i));
                    if (!p)
                        break;
                    i = (int)(static_cast<const uint8_t *>(p) - row);
                }
                const long long c = row + i - mat;
                const int co[3] = {i, j, k};
                for (int a = 0; a < 3; ++a)
                    for (int s = -1; s <= 1; s += 2)
                    {
                        int qq = co[a] + s;
                        if (qq < 0 || qq >= nn[a])
                            continue;
                        long long nb = c + s * dirs[a];
                        if (mat[nb] == 1)
                            continue;
                        if (cnt < cap)
                        {
                            if (cells)
                                cells[cnt] = nb;
                            if (axes)
                                axes[cnt] = a;
                            if (signs)
                                signs[cnt] = s;
                        }
                        ++cnt;
                    }
            }
    return cnt;
}

int64_t tlm_build_huygens(int nx, int ny, int nz, const uint8_t *mat, int o, int64_t *cells,
                          int32_t *axes, int32_t *out_signs, int64_t cap)
{
    if (!mat || o < 2)
        return 0;
    const int nn[3] = {nx, ny, nz};
    if (2 * o + 2 >= nn[0] || 2 * o + 2 >= nn[1] || 2 * o + 2 >= nn[2])
        return 0;
    int64_t cnt = 0;
    auto add = [&](int i, int j, int k, int axis, int sg) {
        long long c = ((long long)k * ny + j) * nx + i;
        if (mat[c] != 0)
            return;
        if (cnt < cap)
        {
            if (cells)
                cells[cnt] = c;
            if (axes)
                axes[cnt] = axis;
            if (out_signs)
                out_signs[cnt] = sg;
        }
        ++cnt;
    };
    int x0 = o, x1 = nx - 1 - o, y0 = o, y1 = ny - 1 - o, z0 = o, z1 = nz - 1 - o;
    for (int k = z0; k <= z1; ++k)
        for (int j = y0; j <= y1; ++j)
        {
            add(x0, j, k, 0, -1);
            add(x1, j, k, 0, +1);
        }
    for (int k = z0; k <= z1; ++k)
        for (int i = x0; i <= x1; ++i)
        {
            add(i, y0, k, 1, -1);
            add(i, y1, k, 1, +1);
        }
    for (int j = y0; j <= y1; ++j)
        for (int i = x0; i <= x1; ++i)
        {
            add(i, j, z0, 2, -1);
            add(i, j, z1, 2, +1);
        }
    return cnt;
}

void tlm_schedule_tables(int type, float f0, float dt, int step0, int nsteps, float gdw, float gdd,
                         float *sv, float *cph, float *sph)
{
    for (int q = 0; q < nsteps; ++q)
    {
        const int n = step0 + q;
        if (sv)
        {
            float val;
            if (type == TLM_WF_GAUSS_DERIV)
            {
                double u = ((double)n - (double)gdd) / (double)gdw;
                val = (float)(-std::sqrt(2.0 * std::exp(1.0)) * u * std::exp(-u * u));
            }
            else
            {
                float t = n * dt;
                float w = 2.0f * (float)M_PI * f0;
                if (type == TLM_WF_CW_RAMPED)
                {
                    float Tr = 3.0f / f0;
                    float r = (t < Tr) ? 0.5f * (1.0f - std::cos((float)M_PI * t / Tr)) : 1.0f;
                    val = r * std::sin(w * t);
                }
                else if (type == TLM_WF_GAUSS_SINE)
                {
                    float tau = 2.0f / f0, t0 = 3.0f * tau;
                    float u = (t - t0) / tau;
                    val = std::exp(-u * u) * std::sin(w * (t - t0));
                }
                else
                {
                    float tau = 0.5f / f0, t0 = 3.0f * tau;
                    float u = (t - t0) / tau;
                    val = std::exp(-u * u);
                }
            }
            sv[q] = val;
        }
        float phase = 2.0f * (float)M_PI * f0 * (n * dt);
        if (cph)
            cph[q] = std::cos(phase);
        if (sph)
            sph[q] = std::sin(phase);
    }
}

void tlm_dft_tables(const double *freqs, int nfreq, double dt, int nsteps, double *ctab,
                    double *stab)
{
    for (int n = 0; n < nsteps; ++n)
        for (int q = 0; q < nfreq; ++q)
        {
            double ph = 2.0 * M_PI * freqs[q] * ((double)n * dt);
            ctab[(size_t)n * nfreq + q] = std::cos(ph);
            stab[(size_t)n * nfreq + q] = std::sin(ph);
        }
}

} // extern "C"
