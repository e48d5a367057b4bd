// TlmBatch.hip - batched execution of many independent TLM grids
// (include/GpuTlmHip.h, tlm_batch_*). No counterpart in the reference, whose
// GPU path runs one grid per OpenGL context.
//
// Members are ordinary contexts (tlm_create / tlm_upload / tlm_set_*), so a
// grid gives the same bits alone and in a batch: the per-cell arithmetic and
// every monitor write are the single-grid code paths, only the launch that
// drives them differs. A tick advances every active member by one step (see
// tlm_batch_kernels.h), two ticks the FP32 members that can by a pair of
// steps; blocks of ticks are captured in a HIP graph.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Wunused-function" // single-grid kernels of the shared header
#include "tlm_batch_kernels.h"
#include "tlm_context.h"
#pragma clang diagnostic pop

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <string>
#include <vector>

namespace {

thread_local std::string g_batch_create_error = "no error";

constexpr int kKinds = 6; // (stubs 0/1) x (PF_F32, PF_F16, PF_BF16)

struct Member
{
    tlm_ctx *c = nullptr;
    int n0 = 0, nend = 0;
    tlm::BatchClock c0 = {}, end = {}; // clock at step n0, and after the last step
    long long launches0 = 0, pairs0 = 0; // the context's counts at step n0
    bool pairs = false;                // takes pairs of steps (tlm::BatchMember)
    char *buf[2] = {nullptr, nullptr};
    float *vs[2] = {nullptr, nullptr};
    long long cells = 0;
    bool range_err = false; // 16-bit storage: a value outgrew its slab scale
};

} // namespace

struct tlm_batch
{
    int dev = 0;
    hipStream_t stream = nullptr;
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    std::string err = "no error";
    std::vector<Member> mem;
    tlm::BatchClock now = {}; // what is queued so far (the device clock after it ran)
    tlm::BatchClock *d_now = nullptr;
    tlm_batch_tuning tune = {1, 4, 0, 32, 4};
    bool dirty = true;
    // device tables, rebuilt when the membership or the tuning changes
    tlm::BatchMember *d_mem = nullptr;
    size_t mem_cap = 0;
    int *d_gmem[kKinds] = {};
    size_t gmem_cap[kKinds] = {};
    int ngroups[kKinds] = {};
    int2 *d_inj = nullptr, *d_mon = nullptr, *d_smax = nullptr;
    size_t inj_cap = 0, mon_cap = 0, smax_cap = 0;
    int ninj = 0, nplan = 0, nmon = 0, nsmax = 0;
    // the parts of members that take pairs: first entries of inj, last ones of
    // mon and gmem
    int ninj_pair = 0, nmon_pair = 0, ngroups_pair[kKinds] = {};
    tlm::PairGroup *d_pgrp[4] = {}; // by stubs (0, 1) and 2 (cells - 1)
    size_t pgrp_cap[4] = {};
    int npgrp[4] = {};
    int2 *d_pmon = nullptr;
    size_t pmon_cap = 0;
    int npmon = 0;
    bool pair_ready = false;
    int wpb = 4;
    // captured blocks of ticks, one by one and in pairs
    hipGraphExec_t gexec[2] = {};
    int glen[2] = {};
};

namespace {

int bfail(tlm_batch *b, int code, const std::string &msg)
{
    if (b)
        b->err = msg;
    else
        g_batch_create_error = msg;
    return code;
}

int bhip(tlm_batch *b, hipError_t e, const char *what)
{
    return bfail(b, e == hipErrorOutOfMemory ? TLM_ERR_NOMEM : TLM_ERR_HIP,
                 std::string(what) + ": " + hipGetErrorString(e));
}

#define BCHK(b, call)                                                                              \
    do                                                                                             \
    {                                                                                              \
        hipError_t e_ = (call);                                                                    \
        if (e_ != hipSuccess)                                                                      \
            return bhip((b), e_, #call);                                                           \
    } while (0)

// Grows a device buffer to hold n elements (contents not kept).
template <class T> int grow(tlm_batch *b, T **p, size_t *cap, size_t n)
{
    if (n <= *cap && *p)
        return TLM_OK;
    if (*p)
        (void)hipFree(*p);
    *p = nullptr;
    const size_t want = std::max<size_t>(n, 1) + std::max<size_t>(n, 1) / 2;
    BCHK(b, hipMalloc((void **)p, want * sizeof(T)));
    *cap = want;
    return TLM_OK;
}

void drop_graph(tlm_batch *b)
{
    for (int k = 0; k < 2; ++k)
    {
        if (b->gexec[k])
            (void)hipGraphExecDestroy(b->gexec[k]);
        b->gexec[k] = nullptr;
        b->glen[k] = 0;
    }
}

int kind_of(const tlm_ctx *c)
{
    return (c->stubs ? 3 : 0) + c->pf;
}

// Current step of a member (clamped to its end).
int member_now(const tlm_batch *b, const Member &m)
{
    return (int)std::min<long long>(m.nend, m.n0 + (b->now.tick - m.c0.tick));
}

// Its current buffers: pulses and stubs by what was queued while it ran.
void member_bufs(const tlm_batch *b, const Member &m, int *buf, int *vs)
{
    const int n = member_now(b, m);
    const tlm::BatchClock &t = n < m.nend ? b->now : m.end;
    *buf = (m.pairs ? (int)(t.launch - m.c0.launch) : n - m.n0) & 1;
    *vs = m.pairs ? (int)(t.pair - m.c0.pair) & 1 : 0;
}

// The context's counts of launches, as of what was queued.
void member_counts(const tlm_batch *b, const Member &m)
{
    const int n = member_now(b, m);
    const tlm::BatchClock &t = n < m.nend ? b->now : m.end;
    m.c->launches = m.launches0 + (m.pairs ? t.launch - m.c0.launch : n - m.n0);
    m.c->pairs = m.pairs0 + (m.pairs ? t.pair - m.c0.pair : 0);
}

// Queued: `count` launches of one tick each, or of two (pairs).
void advance(tlm_batch *b, int count, bool pairs)
{
    const int per = pairs ? 2 : 1;
    for (Member &m : b->mem)
    {
        const int left = m.nend - member_now(b, m);
        if (left > 0 && left <= count * per)
        {
            const int k = left / per; // launches to its end: no pair straddles it
            m.end = {b->now.tick + left, b->now.launch + k, b->now.pair + (pairs ? k : 0)};
        }
    }
    b->now.tick += count * per;
    b->now.launch += count;
    b->now.pair += pairs ? count : 0;
}

// ---- pairs of steps ----

// Whether the batch's launch shape is its own to choose (as pair_active).
bool pairs_wanted(const tlm_batch *b)
{
    const tlm_batch_tuning d = tlm_batch().tune, &t = b->tune;
    return t.planes == d.planes && t.block_waves == d.block_waves && t.grid_blocks == d.grid_blocks;
}

// Makes a member ready for pairs if it can take them.
int member_pairs(tlm_batch *b, Member &m, bool *ok)
{
    tlm_ctx *c = m.c;
    *ok = false;
    if (!b->pair_ready || !pairs_wanted(b) || c->pf != TLM_PULSE_F32 || !c->pair.ok || !tlmi::pair_suits(c) ||
        m.nend - member_now(b, m) < 2)
        return TLM_OK;
    int rc = c->pair_ready ? (int)TLM_OK : tlmi::prepare_pair(c);
    if (rc)
        return bfail(b, rc, c->err);
    if (c->pair_refused)
        return TLM_OK;
    if (c->nuniq > 0)
        tlmi::mark_fold(c, c->stream);
    BCHK(b, hipStreamSynchronize(c->stream));
    *ok = true;
    return TLM_OK;
}

// Tiles of a member: tb blocks beside the rim, as many as a workgroup's waves
// hold, marched over some `slabs` slabs.
void pair_shape(const tlm_ctx *c, int slabs, tlm::PairArgs &a)
{
    constexpr int waves = tlm::kPairBatchThreads / tlm::kWave;
    const int C = tlm::pair_batch_cells(c->nx);
    a = {};
    a.code = c->code;
    a.uair = c->uair;
    a.props = c->props;
    a.nx = c->nx;
    a.ny = c->ny;
    a.nz = c->nz;
    a.Pp = c->Pp;
    a.rho = c->rho;
    a.nmat = std::min(c->nmat, 254);
    a.strips = (int)(c->Pp / tlm::kWave);
    a.hb = (c->nx + tlm::kWave - 1) / tlm::kWave;
    if (a.strips <= C * waves)
        a.hb = 0; // the tile is the slab
    const int most = std::max(C * waves - 2 * a.hb, C), nt = (a.strips + most - 1) / most;
    a.tb = ((a.strips + nt - 1) / nt + C - 1) / C * C;
    a.ntile = (a.strips + a.tb - 1) / a.tb;
    const int nzc = std::max(1, (c->nz + slabs / 2) / slabs);
    a.zc = (c->nz + nzc - 1) / nzc;
    a.mPp = tlm::magic_div((unsigned)c->Pp);
    a.mnx = tlm::magic_div((unsigned)c->nx);
    if (c->nuniq > 0)
        a.fold = tlmi::fold_at(c, 0);
}

// Slabs per tile: 16 where that leaves two tiles a CU or more, else 8 or 4, in
// batches of the smallest grids 2. Us a tick at 16 / by this rule: one grid of
// 64^3 25.2 / 8.7, four of 32 to 64 cells an axis 26.0 / 12.6 (13.2 at 2), 64
// of 16 to 40 62 / 50, 64 of 32 to 128 264 / 264 (10 slabs 262, 32 270); longer
// marches lose in large batches too (six of 200 to 256 806, 863 at 32).
int pair_slabs(const tlm_batch *b)
{
    int slabs = 16;
    for (; slabs > 2; slabs /= 2)
    {
        long long n = 0;
        for (const Member &m : b->mem)
            if (m.pairs)
            {
                tlm::PairArgs a;
                pair_shape(m.c, slabs, a);
                n += (long long)a.ntile * ((a.nz + a.zc - 1) / a.zc);
            }
        if (n >= (slabs == 4 ? 128 : 512))
            break;
    }
    return slabs;
}

// The tiles in launch order: workgroup w runs on XCD w % 8, so the members'
// tiles of a slab range go together to the XCD with the least to do, largest
// first, and an XCD's list is every eighth entry.
std::vector<tlm::PairGroup> pair_order(const std::vector<tlm::BatchMember> &hm, bool stubs, int cells)
{
    struct Unit
    {
        int mem, tz;
        long long cost;
    };
    std::vector<Unit> unit;
    for (size_t i = 0; i < hm.size(); ++i)
    {
        const tlm::PairArgs &a = hm[i].pa;
        if (!hm[i].pairs || (hm[i].vs[0] != nullptr) != stubs || tlm::pair_batch_cells(a.nx) != cells)
            continue;
        for (int z = 0; z * a.zc < a.nz; ++z)
            unit.push_back({(int)i, z, (long long)a.ntile * (a.tb + 2 * a.hb) * (std::min(a.zc, a.nz - z * a.zc) + 2)});
    }
    std::stable_sort(unit.begin(), unit.end(), [](const Unit &x, const Unit &y) { return x.cost > y.cost; });
    std::vector<tlm::PairGroup> list[tlm::kNumXcd];
    long long load[tlm::kNumXcd] = {};
    size_t most = 0;
    for (const Unit &u : unit)
    {
        const int x = (int)(std::min_element(load, load + tlm::kNumXcd) - load);
        load[x] += u.cost;
        for (int t = 0; t < hm[u.mem].pa.ntile; ++t)
            list[x].push_back({u.mem, u.tz, t});
        most = std::max(most, list[x].size());
    }
    std::vector<tlm::PairGroup> out(most * tlm::kNumXcd, tlm::PairGroup{-1, 0, 0});
    for (int x = 0; x < tlm::kNumXcd; ++x)
        for (size_t l = 0; l < list[x].size(); ++l)
            out[l * tlm::kNumXcd + x] = list[x][l];
    return out;
}

// The kernel of a list (tlm_batch::d_pgrp) and its LDS.
using PairKernel = void (*)(const tlm::BatchMember *, const tlm::PairGroup *, tlm::BatchNow, const int2 *,
                            int, int);
PairKernel pair_kernel(int k)
{
    constexpr int NT = tlm::kPairBatchThreads;
    return k == 0   ? tlm::k_step2_batch<false, 1, NT>
           : k == 1 ? tlm::k_step2_batch<true, 1, NT>
           : k == 2 ? tlm::k_step2_batch<false, 2, NT>
                    : tlm::k_step2_batch<true, 2, NT>;
}
int pair_lds(int k)
{
    constexpr int NT = tlm::kPairBatchThreads;
    const int nmat = k & 1 ? 254 : 0;
    return k < 2 ? tlm::pair_lds<1, NT>(nmat) : tlm::pair_lds<2, NT>(nmat);
}

// Rebuilds the member descriptors, the group tables and the monitor entry
// lists. The stream is idle when this runs (tables are read by queued work).
int rebuild(tlm_batch *b)
{
    BCHK(b, hipStreamSynchronize(b->stream));
    drop_graph(b);
    b->wpb = std::max(1, std::min(4, b->tune.block_waves > 0 ? b->tune.block_waves : 4));
    const int wpb = b->wpb;
    std::vector<tlm::BatchMember> hm(b->mem.size());
    std::vector<int> gm[kKinds];
    std::vector<int2> inj, inj1, plan, mon, pmon, smax;
    // first the members that take single steps, then those that take pairs
    std::vector<size_t> order;
    for (bool pairs : {false, true})
        for (size_t i = 0; i < b->mem.size(); ++i)
        {
            Member &M = b->mem[i];
            if (!pairs)
            {
                // from here on the member counts from its present step
                int s = 0, v = 0;
                member_bufs(b, M, &s, &v);
                if (s)
                    std::swap(M.buf[0], M.buf[1]);
                if (v)
                    std::swap(M.vs[0], M.vs[1]);
                member_counts(b, M);
                M.launches0 = M.c->launches;
                M.pairs0 = M.c->pairs;
                M.n0 = member_now(b, M);
                M.c0 = M.end = b->now;
                M.c->A = M.buf[0];
                M.c->B = M.buf[1];
                if (M.pairs)
                {
                    M.c->Vs = M.vs[0];
                    M.c->Vs2 = M.vs[1];
                }
                int rc = member_pairs(b, M, &M.pairs);
                if (rc)
                    return rc;
                M.vs[0] = M.c->Vs;
                M.vs[1] = M.pairs ? M.c->Vs2 : nullptr;
            }
            if (M.pairs == pairs)
                order.push_back(i);
        }
    for (int k = 0; k < kKinds; ++k)
        b->ngroups_pair[k] = 0;
    b->nmon_pair = 0;
    const int slabs = pair_slabs(b);
    for (size_t i : order)
    {
        const Member &M = b->mem[i];
        tlm_ctx *c = M.c;
        tlm::BatchMember &d = hm[i];
        d = {};
        const int pl = c->pf == TLM_PULSE_F32 ? b->tune.planes : b->tune.planes16;
        const int zc = pl > 0 ? std::min(pl, c->nz) : c->nz;
        const int nzc = (c->nz + zc - 1) / zc;
        const int strips = (int)(c->Pp / tlm::kWave);
        const int tasks = strips * nzc;
        const int groups = (tasks + wpb - 1) / wpb;
        tlm::StepArgs &a = d.st;
        a.A = nullptr;
        a.B = nullptr;
        a.Vs = c->Vs;
        a.code = c->code;
        a.uair = c->uair;
        a.props = c->props;
        a.epart = nullptr;
        a.slab = c->slab;
        a.dsc = nullptr;
        a.esc = nullptr;
        a.mpart = c->mpart;
        a.nx = c->nx;
        a.ny = c->ny;
        a.nz = c->nz;
        a.nxy = (int)c->nxy;
        a.Pp = c->Pp;
        a.P = c->P;
        a.PB = c->PB;
        a.h0 = c->h0;
        a.h1 = c->h1;
        a.strips = strips;
        a.zc = zc;
        a.nzc = nzc;
        a.tasks = tasks;
        a.groups = groups;
        a.rho = c->rho;
        a.nmat = c->nmat;
        a.mstrips = tlm::magic_div((unsigned)strips);
        a.mPp = tlm::magic_div((unsigned)c->Pp);
        a.mnx = tlm::magic_div((unsigned)c->nx);
        d.buf[0] = M.buf[0];
        d.buf[1] = M.buf[1];
        d.vs[0] = M.vs[0];
        d.vs[1] = M.vs[1];
        d.c0 = M.c0;
        d.pairs = M.pairs;
        if (M.pairs)
            pair_shape(c, slabs, d.pa);
        d.n0 = M.n0;
        d.nend = M.nend;
        d.pf = c->pf;
        d.sbase = c->base;
        for (int q = 0; q < 2; ++q)
        {
            d.scl[q] = c->scl[q];
            d.iscl[q] = c->iscl[q];
        }
        d.ucell = c->ucell;
        d.ubeg = c->ubeg;
        d.spol = c->spol;
        d.samp = c->samp;
        d.sv = c->sv;
        d.nsched = c->nsteps;
        d.mreg = c->mreg;
        d.qinj = c->qinj;
        d.flag = c->flag;
        d.rp = std::max(1.0f, std::fabs(c->rho));
        d.fmax = tlmi::format_max(c->pf);
        d.prcell = c->prcell;
        d.prrec = c->prrec;
        d.npr = c->npr;
        d.inv_dl = c->inv_dl;
        d.pcells = c->pcells;
        d.ploop = c->ploop;
        d.poff = c->poff;
        d.ppol = c->ppol;
        d.prec = c->prec;
        d.np = c->np;
        const int k = kind_of(c);
        d.group0 = (int)gm[k].size();
        gm[k].insert(gm[k].end(), groups, (int)i);
        for (int u = 0; u < c->nuniq; ++u)
            (M.pairs ? inj : inj1).push_back(make_int2((int)i, u));
        if (M.pairs)
        {
            b->ngroups_pair[k] += groups;
            b->nmon_pair += c->npr + c->np;
            for (int w = 0; w < (c->npr + 7) / 8 + c->np; ++w)
                pmon.push_back(make_int2((int)i, w));
        }
        if (c->pf != TLM_PULSE_F32)
            for (int z = 0; z < c->nz; ++z)
            {
                plan.push_back(make_int2((int)i, z));
                smax.push_back(make_int2((int)i, z));
            }
        for (int p = 0; p < c->npr + c->np; ++p)
            mon.push_back(make_int2((int)i, p));
    }
    b->ninj_pair = (int)inj.size();
    inj.insert(inj.end(), inj1.begin(), inj1.end());
    b->ninj = (int)inj.size();
    b->nplan = (int)plan.size();
    inj.insert(inj.end(), plan.begin(), plan.end());
    b->nmon = (int)mon.size();
    b->nsmax = (int)smax.size();
    int rc;
    if ((rc = grow(b, &b->d_mem, &b->mem_cap, hm.size())) ||
        (rc = grow(b, &b->d_inj, &b->inj_cap, inj.size())) ||
        (rc = grow(b, &b->d_mon, &b->mon_cap, mon.size())) ||
        (rc = grow(b, &b->d_smax, &b->smax_cap, smax.size())))
        return rc;
    if (!hm.empty())
        BCHK(b, hipMemcpy(b->d_mem, hm.data(), hm.size() * sizeof(hm[0]), hipMemcpyHostToDevice));
    if (!inj.empty())
        BCHK(b, hipMemcpy(b->d_inj, inj.data(), inj.size() * sizeof(int2), hipMemcpyHostToDevice));
    if (!mon.empty())
        BCHK(b, hipMemcpy(b->d_mon, mon.data(), mon.size() * sizeof(int2), hipMemcpyHostToDevice));
    if (!smax.empty())
        BCHK(b, hipMemcpy(b->d_smax, smax.data(), smax.size() * sizeof(int2),
                          hipMemcpyHostToDevice));
    for (int k = 0; k < kKinds; ++k)
    {
        b->ngroups[k] = (int)gm[k].size();
        if (gm[k].empty())
            continue;
        if ((rc = grow(b, &b->d_gmem[k], &b->gmem_cap[k], gm[k].size())))
            return rc;
        BCHK(b, hipMemcpy(b->d_gmem[k], gm[k].data(), gm[k].size() * sizeof(int),
                          hipMemcpyHostToDevice));
    }
    for (int k = 0; k < 4; ++k)
    {
        const std::vector<tlm::PairGroup> g = pair_order(hm, k & 1, 1 + k / 2);
        b->npgrp[k] = (int)g.size();
        if (g.empty())
            continue;
        if ((rc = grow(b, &b->d_pgrp[k], &b->pgrp_cap[k], g.size())))
            return rc;
        BCHK(b, hipMemcpy(b->d_pgrp[k], g.data(), g.size() * sizeof(g[0]), hipMemcpyHostToDevice));
    }
    b->npmon = (int)pmon.size();
    if (!pmon.empty())
    {
        if ((rc = grow(b, &b->d_pmon, &b->pmon_cap, pmon.size())))
            return rc;
        BCHK(b, hipMemcpy(b->d_pmon, pmon.data(), pmon.size() * sizeof(int2), hipMemcpyHostToDevice));
    }
    b->dirty = false;
    return TLM_OK;
}

// One kind's step launch over its first ng groups; nmon > 0 appends the
// workgroups that take the first nmon records of the tick.
template <bool S, int PF> void launch_kind(tlm_batch *b, int k, int ng, int nmon, const tlm::BatchNow &now)
{
    const int blocks = b->tune.grid_blocks > 0 ? std::min(ng, b->tune.grid_blocks) : ng;
    const int bt = b->wpb * tlm::kWave;
    const int mon_blocks = (nmon + bt - 1) / bt;
    hipLaunchKernelGGL((tlm::k_step_batch<S, PF>), dim3(blocks + mon_blocks), dim3(bt), 0,
                       b->stream, b->d_mem, b->d_gmem[k], ng, now, b->d_mon, nmon,
                       blocks);
}

// One tick of all members, or of those that do not take pairs, `off` after the
// device clock.
void queue_tick(tlm_batch *b, bool all, tlm::BatchClock off)
{
    const tlm::BatchNow now{b->d_now, off};
    const int skip = all ? 0 : b->ninj_pair, ninj = b->ninj - skip;
    if (ninj + b->nplan > 0)
    {
        const int n = ninj + b->nplan, t = 128;
        hipLaunchKernelGGL(tlm::k_inject_batch, dim3((n + t - 1) / t), dim3(t), 0, b->stream,
                           b->d_mem, b->d_inj + skip, ninj, b->nplan, now);
    }
    // the records ride with the first kind that has members
    int mon = b->nmon - (all ? 0 : b->nmon_pair);
    auto kind = [&](int k, auto launch) {
        const int ng = b->ngroups[k] - (all ? 0 : b->ngroups_pair[k]);
        if (!ng)
            return;
        launch(k, ng, mon);
        mon = 0;
    };
    kind(0, [&](int k, int ng, int m) { launch_kind<false, tlm::PF_F32>(b, k, ng, m, now); });
    kind(1, [&](int k, int ng, int m) { launch_kind<false, tlm::PF_F16>(b, k, ng, m, now); });
    kind(2, [&](int k, int ng, int m) { launch_kind<false, tlm::PF_BF16>(b, k, ng, m, now); });
    kind(3, [&](int k, int ng, int m) { launch_kind<true, tlm::PF_F32>(b, k, ng, m, now); });
    kind(4, [&](int k, int ng, int m) { launch_kind<true, tlm::PF_F16>(b, k, ng, m, now); });
    kind(5, [&](int k, int ng, int m) { launch_kind<true, tlm::PF_BF16>(b, k, ng, m, now); });
    if (mon > 0)
    {
        // no member with step groups (cannot happen with active members):
        // the records alone, through an empty step grid
        launch_kind<false, tlm::PF_F32>(b, 0, 0, mon, now);
    }
    if (b->nsmax > 0)
        hipLaunchKernelGGL(tlm::k_slab_max_batch, dim3(b->nsmax), dim3(256), 0, b->stream,
                           b->d_mem, b->d_smax, now);
}

// Two ticks: the members that take pairs in one launch, then the others' two.
void queue_pair(tlm_batch *b, tlm::BatchClock off)
{
    constexpr int NT = tlm::kPairBatchThreads;
    int mon = b->npmon;
    for (int k = 0; k < 4; ++k)
    {
        if (!b->npgrp[k])
            continue;
        hipLaunchKernelGGL(pair_kernel(k),
                           dim3(b->npgrp[k] + (mon + NT / tlm::kWave - 1) / (NT / tlm::kWave)), dim3(NT),
                           pair_lds(k), b->stream, b->d_mem, b->d_pgrp[k], tlm::BatchNow{b->d_now, off}, b->d_pmon, mon,
                           b->npgrp[k]);
        mon = 0;
    }
    int single = b->ninj - b->ninj_pair + b->nplan;
    for (int k = 0; k < kKinds; ++k)
        single += b->ngroups[k] - b->ngroups_pair[k];
    if (!single)
        return;
    queue_tick(b, false, off);
    ++off.tick;
    queue_tick(b, false, off);
}

// Queues `count` ticks, or pairs of ticks, in captured blocks of the tuning's
// length as far as they go.
int queue_blocks(tlm_batch *b, int count, bool pairs)
{
    const tlm::BatchClock per = pairs ? tlm::BatchClock{2, 1, 1} : tlm::BatchClock{1, 1, 0};
    auto times = [&](int t) { return tlm::BatchClock{per.tick * t, per.launch * t, per.pair * t}; };
    auto block = [&](int len) {
        for (int t = 0; t < len; ++t)
            if (pairs)
                queue_pair(b, times(t));
            else
                queue_tick(b, true, times(t));
        hipLaunchKernelGGL(tlm::k_tick, dim3(1), dim3(64), 0, b->stream, b->d_now, times(len));
    };
    const int k = pairs ? 1 : 0, L = pairs ? b->tune.graph_ticks / 2 : b->tune.graph_ticks;
    int left = count;
    if (L > 0 && left >= L)
    {
        if (!b->gexec[k] || b->glen[k] != L)
        {
            if (b->gexec[k])
                (void)hipGraphExecDestroy(b->gexec[k]);
            b->gexec[k] = nullptr;
            hipGraph_t g = nullptr;
            BCHK(b, hipStreamBeginCapture(b->stream, hipStreamCaptureModeThreadLocal));
            block(L);
            BCHK(b, hipStreamEndCapture(b->stream, &g));
            hipError_t e = hipGraphInstantiate(&b->gexec[k], g, nullptr, nullptr, 0);
            (void)hipGraphDestroy(g);
            if (e != hipSuccess)
            {
                b->gexec[k] = nullptr;
                return bhip(b, e, "hipGraphInstantiate");
            }
            b->glen[k] = L;
        }
        while (left >= L)
        {
            BCHK(b, hipGraphLaunch(b->gexec[k], b->stream));
            left -= L;
        }
    }
    if (left > 0)
        block(left);
    BCHK(b, hipGetLastError());
    advance(b, count, pairs);
    return TLM_OK;
}

int queue_ticks(tlm_batch *b, int nticks)
{
    if (b->dirty)
    {
        int rc = rebuild(b);
        if (rc)
            return rc;
    }
    for (int left = nticks; left > 0;)
    {
        // as many pairs as end at no member's odd step; with none, a single
        // tick; without members that take pairs, single ticks throughout
        int count = left / 2;
        bool any = false;
        for (const Member &m : b->mem)
        {
            const int r = m.nend - member_now(b, m);
            if (!m.pairs || r <= 0)
                continue;
            any = true;
            if (r % 2)
                count = std::min(count, r / 2);
        }
        const bool pairs = any && count > 0;
        if (!pairs)
            count = any ? 1 : left;
        int rc = queue_blocks(b, count, pairs);
        if (rc)
            return rc;
        left -= pairs ? 2 * count : count;
    }
    return TLM_OK;
}

// Waits for the queued ticks and brings every member's host-side state up
// to date (current pulse buffer, step counters, running probe DFT). A 16-bit
// member whose range flag is set is marked (its results are invalid); the
// others go on, and tlm_batch_remove reports it for that member only.
int sync_members(tlm_batch *b)
{
    BCHK(b, hipSetDevice(b->dev));
    BCHK(b, hipStreamSynchronize(b->stream));
    for (Member &m : b->mem)
    {
        tlm_ctx *c = m.c;
        const int now = member_now(b, m);
        int s = 0, v = 0;
        member_bufs(b, m, &s, &v);
        c->A = m.buf[s];
        c->B = m.buf[s ^ 1];
        if (m.pairs)
        {
            c->Vs = m.vs[v];
            c->Vs2 = m.vs[v ^ 1];
        }
        member_counts(b, m);
        c->next_step = now;
        c->steps_run_hi = std::max(c->steps_run_hi, now);
        if (c->npr > 0 && c->nfreq > 0 && c->dft_done < now)
            tlmi::queue_probe_dft(c, c->dft_done, now, b->stream);
        if (c->flag && !m.range_err)
        {
            int f = 0;
            BCHK(b, hipMemcpy(&f, c->flag, sizeof(int), hipMemcpyDeviceToHost));
            m.range_err = f != 0;
        }
    }
    BCHK(b, hipStreamSynchronize(b->stream));
    return TLM_OK;
}

// Ticks for timing a launch shape, `ticks` or so: as many as go in whole pairs
// where members take pairs (single ticks among them, as at a member's odd end,
// would be timed for the shape that takes pairs as for one that does not); 0 if
// a member has to end first.
int pair_window(const tlm_batch *b, int ticks)
{
    int even = ticks + ticks % 2;
    bool any = false;
    for (const Member &m : b->mem)
    {
        const int r = m.nend - member_now(b, m);
        if (!m.pairs || r <= 0)
            continue;
        any = true;
        if (r % 2)
            even = std::min(even, r - 1);
    }
    return any ? even : ticks;
}

long long active_cells(const tlm_batch *b)
{
    long long n = 0;
    for (const Member &m : b->mem)
        if (member_now(b, m) < m.nend)
            n += m.cells;
    return n;
}

} // namespace

extern "C" {

int tlm_batch_create(int device, tlm_batch **out)
{
    if (!out)
        return bfail(nullptr, TLM_ERR_ARG, "tlm_batch_create: out is NULL");
    *out = nullptr;
    if (device < 0 || device >= tlm_device_count())
        return bfail(nullptr, TLM_ERR_NO_DEVICE, "no such HIP device");
    tlm_batch *b = new tlm_batch;
    b->dev = device;
    auto bail = [&](hipError_t e, const char *what) {
        bhip(b, e, what);
        g_batch_create_error = b->err;
        tlm_batch_destroy(b);
        return e == hipErrorOutOfMemory ? TLM_ERR_NOMEM : TLM_ERR_HIP;
    };
    hipError_t e;
    if ((e = hipSetDevice(device)) != hipSuccess)
        return bail(e, "hipSetDevice");
    if ((e = hipStreamCreateWithFlags(&b->stream, hipStreamNonBlocking)) != hipSuccess)
        return bail(e, "hipStreamCreate");
    if ((e = hipEventCreate(&b->ev0)) != hipSuccess || (e = hipEventCreate(&b->ev1)) != hipSuccess)
        return bail(e, "hipEventCreate");
    if ((e = hipMalloc((void **)&b->d_now, sizeof(tlm::BatchClock))) != hipSuccess)
        return bail(e, "hipMalloc");
    if ((e = hipMemset(b->d_now, 0, sizeof(tlm::BatchClock))) != hipSuccess)
        return bail(e, "hipMemset");
    b->pair_ready = true;
    for (int k = 0; k < 4; ++k)
        if (hipFuncSetAttribute((const void *)pair_kernel(k), hipFuncAttributeMaxDynamicSharedMemorySize,
                                pair_lds(k)) != hipSuccess)
        {
            (void)hipGetLastError();
            b->pair_ready = false;
        }
    *out = b;
    return TLM_OK;
}

void tlm_batch_destroy(tlm_batch *b)
{
    if (!b)
        return;
    (void)hipSetDevice(b->dev);
    if (b->stream)
        (void)hipStreamSynchronize(b->stream);
    for (Member &m : b->mem)
        m.c->batch = nullptr;
    b->mem.clear();
    drop_graph(b);
    for (void *p : {(void *)b->d_now, (void *)b->d_mem, (void *)b->d_inj, (void *)b->d_mon,
                    (void *)b->d_smax, (void *)b->d_pmon, (void *)b->d_pgrp[0], (void *)b->d_pgrp[1],
                    (void *)b->d_pgrp[2], (void *)b->d_pgrp[3]})
        if (p)
            (void)hipFree(p);
    for (int k = 0; k < kKinds; ++k)
        if (b->d_gmem[k])
            (void)hipFree(b->d_gmem[k]);
    for (hipEvent_t ev : {b->ev0, b->ev1})
        if (ev)
            (void)hipEventDestroy(ev);
    if (b->stream)
        (void)hipStreamDestroy(b->stream);
    delete b;
}

const char *tlm_batch_last_error(const tlm_batch *b)
{
    return b ? b->err.c_str() : g_batch_create_error.c_str();
}

int tlm_batch_add(tlm_batch *b, tlm_ctx *c, int nsteps)
{
    if (!b || !c || nsteps < 0)
        return bfail(b, TLM_ERR_ARG, "tlm_batch_add: bad arguments");
    if (c->batch)
        return bfail(b, TLM_ERR_STATE, "context is already a batch member");
    if (c->dev != b->dev)
        return bfail(b, TLM_ERR_ARG, "context and batch are on different devices");
    if (!c->uploaded || !c->sv)
        return bfail(b, TLM_ERR_STATE, "batch member needs tlm_upload and tlm_set_schedule first");
    if (c->nf > 0 || c->nh > 0 || c->pa >= 0 || c->frame_every > 0)
        return bfail(b, TLM_ERR_UNSUPPORTED,
                     "batch members record probes and ports (no Js, Huygens, plane or frames)");
    if (c->every > 0)
        return bfail(b, TLM_ERR_UNSUPPORTED,
                     "batch members record no energy: tlm_set_energy_every(ctx, 0) before joining");
    const int n0 = c->next_step;
    if (n0 + nsteps > c->nsteps)
        return bfail(b, TLM_ERR_ARG, "steps beyond the member's schedule");
    if (c->npr > 0 && c->nfreq > 0 && c->dft_done != n0)
        return bfail(b, TLM_ERR_STATE, "probe DFT needs contiguous steps");
    BCHK(b, hipSetDevice(b->dev));
    BCHK(b, hipStreamSynchronize(c->stream));
    if (c->pf != TLM_PULSE_F32 && !c->materialized)
    {
        int rc = tlmi::materialize(c, n0);
        if (rc)
            return bfail(b, rc, c->err);
    }
    Member m;
    m.c = c;
    m.n0 = n0;
    m.nend = n0 + nsteps;
    m.c0 = m.end = b->now;
    m.buf[0] = c->A;
    m.buf[1] = c->B;
    m.vs[0] = c->Vs;
    m.launches0 = c->launches;
    m.pairs0 = c->pairs;
    m.cells = (long long)c->nx * c->ny * c->nz;
    b->mem.push_back(m);
    c->batch = b;
    b->dirty = true;
    return TLM_OK;
}

int tlm_batch_remove(tlm_batch *b, tlm_ctx *c)
{
    if (!b || !c)
        return bfail(b, TLM_ERR_ARG, "tlm_batch_remove: bad arguments");
    auto it = std::find_if(b->mem.begin(), b->mem.end(), [&](const Member &m) { return m.c == c; });
    if (it == b->mem.end())
        return bfail(b, TLM_ERR_ARG, "context is not a member of this batch");
    int rc = sync_members(b);
    const bool range_err = it->range_err;
    b->mem.erase(it);
    c->batch = nullptr;
    b->dirty = true;
    if (rc == TLM_OK && range_err)
    {
        tlmi::fail(c, TLM_ERR_RANGE, "16-bit pulse storage: a value exceeded the range its slab scale allows");
        return bfail(b, TLM_ERR_RANGE,
                     "this member's 16-bit pulse storage exceeded its slab scale: its results are "
                     "invalid (the other members are not affected)");
    }
    return rc;
}

int tlm_batch_run(tlm_batch *b, int nticks)
{
    if (!b || nticks < 0)
        return bfail(b, TLM_ERR_ARG, "tlm_batch_run: bad arguments");
    if (nticks == 0 || b->mem.empty())
        return TLM_OK;
    BCHK(b, hipSetDevice(b->dev));
    return queue_ticks(b, nticks);
}

int tlm_batch_sync(tlm_batch *b)
{
    if (!b)
        return TLM_ERR_ARG;
    return sync_members(b);
}

int tlm_batch_members(tlm_batch *b, tlm_ctx **members, int32_t *remaining, int cap)
{
    if (!b || cap < 0)
        return TLM_ERR_ARG;
    const int n = (int)b->mem.size();
    for (int i = 0; i < n && i < cap; ++i)
    {
        if (members)
            members[i] = b->mem[i].c;
        if (remaining)
            remaining[i] = b->mem[i].nend - member_now(b, b->mem[i]);
    }
    return n;
}

int tlm_batch_set_tuning(tlm_batch *b, const tlm_batch_tuning *t)
{
    if (!b || !t || t->planes < 0 || t->block_waves < 0 || t->block_waves > 4 ||
        t->grid_blocks < 0 || t->graph_ticks < 0 || t->planes16 < 0)
        return bfail(b, TLM_ERR_ARG, "tlm_batch_set_tuning: bad tuning");
    b->tune = *t;
    b->dirty = true;
    return TLM_OK;
}

int tlm_batch_get_tuning(const tlm_batch *b, tlm_batch_tuning *t)
{
    if (!b || !t)
        return TLM_ERR_ARG;
    *t = b->tune;
    return TLM_OK;
}

int tlm_batch_time(tlm_batch *b, int nticks, float *ms, int64_t *cell_updates)
{
    if (!b || nticks <= 0)
        return bfail(b, TLM_ERR_ARG, "tlm_batch_time: bad arguments");
    BCHK(b, hipSetDevice(b->dev));
    if (b->dirty)
    {
        int rc = rebuild(b);
        if (rc)
            return rc;
    }
    long long cu = 0;
    for (const Member &m : b->mem)
    {
        const long long now = member_now(b, m);
        cu += m.cells * std::max<long long>(0, std::min<long long>(m.nend - now, nticks));
    }
    BCHK(b, hipEventRecord(b->ev0, b->stream));
    int rc = queue_ticks(b, nticks);
    if (rc)
        return rc;
    BCHK(b, hipEventRecord(b->ev1, b->stream));
    BCHK(b, hipEventSynchronize(b->ev1));
    float t = 0.f;
    BCHK(b, hipEventElapsedTime(&t, b->ev0, b->ev1));
    if (ms)
        *ms = t;
    if (cell_updates)
        *cell_updates = cu;
    return TLM_OK;
}

// Online autotuner: every candidate (slabs per wave task x waves per
// workgroup x grid) runs real ticks of the batch (the launch shape never
// changes results), timed with events; the fastest per active cell wins.
int tlm_batch_autotune(tlm_batch *b, int ticks_per_candidate, tlm_batch_tuning *best)
{
    if (!b || ticks_per_candidate <= 0)
        return bfail(b, TLM_ERR_ARG, "tlm_batch_autotune: bad arguments");
    if (b->mem.empty())
        return bfail(b, TLM_ERR_STATE, "tlm_batch_autotune: empty batch");
    const tlm_batch_tuning keep = b->tune;
    bool have16 = false, have32 = false;
    for (const Member &m : b->mem)
        (m.c->pf == TLM_PULSE_F32 ? have32 : have16) = true;
    std::vector<tlm_batch_tuning> cands;
    for (int p : {1, 2, 4, 8})
        for (int w : {2, 4})
            for (int g : {0, 2048})
                for (int p16 : {2, 4, 8})
                {
                    if ((!have32 && p != 1) || (!have16 && p16 != 4))
                        continue;
                    cands.push_back({p, w, g, 0, p16});
                }
    tlm_batch_tuning top = keep;
    double top_ns = 1e300;
    for (const tlm_batch_tuning &t : cands)
    {
        if (active_cells(b) == 0)
            break;
        b->tune = t;
        b->dirty = true;
        float ms = 0.f;
        int64_t cu = 0;
        int rc = tlm_batch_time(b, pairs_wanted(b) ? 2 : 1, &ms, &cu); // warm-up (tables, the kernel's first run)
        int window = ticks_per_candidate;
        while (!rc && (window = pair_window(b, ticks_per_candidate)) == 0)
            rc = tlm_batch_time(b, 1, &ms, &cu);
        if (!rc)
            rc = tlm_batch_time(b, window, &ms, &cu);
        if (rc)
        {
            b->tune = keep;
            b->dirty = true;
            return rc;
        }
        const double ns = cu > 0 ? ms * 1e6 / (double)cu : 1e300;
        if (ns < top_ns)
        {
            top_ns = ns;
            top = t;
        }
    }
    top.graph_ticks = keep.graph_ticks;
    b->tune = top;
    b->dirty = true;
    if (best)
        *best = top;
    return TLM_OK;
}

} // extern "C"
