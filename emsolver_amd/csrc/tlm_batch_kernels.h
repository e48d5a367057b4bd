// tlm_batch_kernels.h - kernels of the batched step: many independent grids
// advanced by the same launches.
//
// Each member grid keeps its own context buffers (pulses, stubs, cell codes,
// monitors). A tick advances every active member by one step: one
// injection launch for all members' soft sources (with the 16-bit scale
// planning), one fused step launch per member kind (stubs x storage format)
// over the concatenated task groups of its members (the first of them also
// taking every member's probe and port records in extra workgroups), one
// slab-maximum launch for the 16-bit members; a one-thread launch advances the
// device clock at the end of a block of ticks. Every launch reads the
// clock from device memory, so a block of ticks can be captured once in a
// HIP graph and replayed. FP32 members take two ticks in one launch
// (k_step2_batch), in which their sources are added, where they can.
#pragma once

#include "tlm_kernels.h"
#include "tlm_step2.h"

namespace tlm {

// Ticks done, step launches done (a pair of ticks is one), pairs among them.
struct BatchClock
{
    long long tick, launch, pair;
};
// Time of a launch: the device clock, and what the block of ticks it belongs to
// did before it. The clock goes on once a block: with a k_tick after each pair of
// ticks one grid of 64^3 took 17.8 us a pair, 15.9 so; 16 of 32 to 128 cells an
// axis 151 and 148.
struct BatchNow
{
    const BatchClock *base;
    BatchClock off;
    __device__ __forceinline__ BatchClock operator()() const
    {
        return {base->tick + off.tick, base->launch + off.launch, base->pair + off.pair};
    }
};

struct BatchMember
{
    StepArgs st;        // geometry and pointers; A/B and the scales are picked per tick
    PairArgs pa;        // the same for pairs of steps
    int pairs;          // the member takes pairs: its buffers alternate by launches
    BatchClock c0;      // the clock at which the member runs its step n0 ...
    char *buf[2];       // ... and pulse buffers: buf[0] holds the incident pulses of that step
    float *vs[2];       // its stubs likewise, by pairs
    int n0, nend;       // the member runs steps [n0, nend) in the batch
    int pf;             // PF_*
    int sbase;          // 16-bit: step whose scales are in buffer 0
    float *scl[2], *iscl[2];
    // soft sources
    const long long *ucell;
    const int *ubeg, *spol;
    const float *samp;
    const float *sv;    // schedule (nsched steps)
    int nsched;
    // 16-bit scale planning
    float *mreg;
    const float *qinj;
    int *flag;
    float rp, fmax;
    // probes and ports
    const long long *prcell;
    float *prrec;
    int npr;
    float inv_dl;
    const long long *pcells, *ploop;
    const int *poff, *ppol;
    float *prec;
    int np;
    int group0;         // first task group of the member in its kind's table
};

// Step of member m at batch time t; >= nend once it has finished.
__device__ __forceinline__ int member_step(const BatchMember &m, const BatchClock &t)
{
    return m.n0 + (int)(t.tick - m.c0.tick);
}
// Buffer with the incident pulses of step n.
__device__ __forceinline__ int member_buf(const BatchMember &m, int n, const BatchClock &t)
{
    return (m.pairs ? (int)(t.launch - m.c0.launch) : n - m.n0) & 1;
}
__device__ __forceinline__ int member_vs(const BatchMember &m, const BatchClock &t)
{
    return m.pairs ? (int)(t.pair - m.c0.pair) & 1 : 0;
}

__device__ __forceinline__ PulseView member_view(const BatchMember &m, int n, const BatchClock &t)
{
    PulseView v;
    v.base = m.buf[member_buf(m, n, t)];
    v.PB = m.st.PB;
    v.Pp = m.st.Pp;
    v.mPp = m.st.mPp;
    v.pf = m.pf;
    v.slab = m.st.slab;
    v.h0 = m.st.h0;
    v.h1 = m.st.h1;
    const int cur = (n - m.sbase) & 1;
    v.sc = m.pf != PF_F32 ? m.scl[cur] : nullptr;
    v.isc = m.pf != PF_F32 ? m.iscl[cur] : nullptr;
    return v;
}

// Injection of every member's soft sources (entries (member, unique cell)),
// then the 16-bit scale planning (entries (member, slab)).
static __global__ void k_inject_batch(const BatchMember *mem, const int2 *ent, int ninj, int nplan,
                               BatchNow now)
{
    const int id = blockIdx.x * blockDim.x + threadIdx.x;
    if (id >= ninj + nplan)
        return;
    const int2 e = ent[id];
    const BatchMember &m = mem[e.x];
    const int n = member_step(m, now());
    if (n >= m.nend)
        return;
    if (id < ninj)
    {
        const PulseView pv = member_view(m, n, now());
        const float over =
            inject_cell(pv, m.ucell[e.y], m.ubeg[e.y], m.ubeg[e.y + 1], m.spol, m.samp, m.sv[n]);
        if (m.pf != PF_F32 && over > m.fmax)
            m.flag[0] = 1;
        return;
    }
    const int cur = (n - m.sbase) & 1;
    PlanArgs pl;
    pl.nz = m.st.nz;
    pl.mreg = m.mreg;
    pl.Q = m.qinj;
    pl.slab = m.st.slab;
    pl.sv = m.sv;
    pl.n = n;
    pl.nsteps = m.nsched;
    pl.rp = m.rp;
    pl.fmax = m.fmax;
    pl.isc_cur = m.iscl[cur];
    pl.sc_next = m.scl[cur ^ 1];
    pl.isc_next = m.iscl[cur ^ 1];
    pl.flag = m.flag;
    plan_slab(pl, e.y, pl.mreg + e.y);
}

// Probe and port records of every member (entries (member, index): index <
// npr is a probe, the rest ports).
__device__ __forceinline__ void monitor_batch_item(const BatchMember *mem, const int2 *ent, int nent,
                                                   BatchNow now, int id)
{
    if (id >= nent)
        return;
    const int2 e = ent[id];
    const BatchMember &m = mem[e.x];
    const int n = member_step(m, now());
    if (n >= m.nend)
        return;
    const PulseView pv = member_view(m, n, now());
    auto take = [&](auto pf) {
        constexpr int PF = decltype(pf)::value;
        if (e.y < m.npr)
            monitor_probe<PF>(pv, e.y, n, m.npr, m.prcell, m.inv_dl, m.prrec);
        else
            monitor_port<PF>(pv, e.y - m.npr, n, m.np, m.pcells, m.poff, m.ppol, m.ploop, m.prec);
    };
    if (m.pf == PF_F32)
        take(std::integral_constant<int, PF_F32>{});
    else if (m.pf == PF_F16)
        take(std::integral_constant<int, PF_F16>{});
    else
        take(std::integral_constant<int, PF_BF16>{});
}

// Fused scatter + connect for the members of one kind. gmem[g] is the member
// of task group g; the workgroups walk the groups in XCD-contiguous ranges
// (a persistent grid when there are fewer workgroups than groups).
// Workgroups from mon_from on take the tick's probe and port records of all
// members (they read the incident pulses, which the step only reads).
template <bool STUBS, int PF>
__global__ void __launch_bounds__(256) k_step_batch(const BatchMember *mem, const int *gmem,
                                                    int ngroups, BatchNow now,
                                                    const int2 *ment, int nment, int mon_from)
{
    if ((int)blockIdx.x >= mon_from)
    {
        monitor_batch_item(mem, ment, nment, now,
                           ((int)blockIdx.x - mon_from) * (int)blockDim.x + (int)threadIdx.x);
        return;
    }
    const int lane = threadIdx.x & (kWave - 1);
    const int wpb = blockDim.x / kWave;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const BatchClock t = now();
    const XcdRange gr = xcd_range(blockIdx.x, mon_from, ngroups);
    for (int g = gr.first; g < gr.end; g += gr.step)
    {
        const int mi = gmem[g];
        const BatchMember &m = mem[mi];
        const int n = member_step(m, t);
        if (n >= m.nend)
            continue;
        const int task = (g - m.group0) * wpb + wave;
        if (task >= m.st.tasks)
            continue;
        StepArgs a = m.st;
        const int s = member_buf(m, n, t);
        a.A = m.buf[s];
        a.B = m.buf[s ^ 1];
        a.Vs = m.vs[member_vs(m, t)];
        if (PF != PF_F32)
        {
            const int cur = (n - m.sbase) & 1;
            a.dsc = m.scl[cur];
            a.esc = m.iscl[cur ^ 1];
        }
        if constexpr (PF == PF_F32)
            strip_task<STUBS, false, false, PF>(a, task, lane);
        else
            strip_task16<STUBS, false, PF>(a, task, lane);
    }
}

// Threads of the pairs' tiles; blocks per wave (C): one, two where the rim of
// one row on either side is wide. 64 grids of 32 to 128 cells an axis (21.2 M
// cells), us a tick: 264 with one block in each of 16 waves, 277 of 8 waves;
// two blocks 295 of 16 waves and 297 of 8. One / two blocks: 24 grids of 128 to
// 200 1078 / 1106, six of 200 to 256 806 / 773, four of 300 to 330 1959 / 1374.
constexpr int kPairBatchThreads = 1024;
__host__ __device__ inline int pair_batch_cells(int nx)
{
    return nx > 192 ? 2 : 1;
}

// A place in the launch of pairs: tile (tz, tt) of a member; member -1: none.
struct PairGroup
{
    int mem, tz, tt;
};

// Steps n and n+1 of the FP32 members of one kind that take pairs, one tile
// per workgroup (k_step2). Workgroups from mon_from on take both steps'
// probe and port records, a wave each (ment: member, wave).
template <bool STUBS, int C, int NT>
__global__ void __launch_bounds__(NT, kPairOcc)
    k_step2_batch(const BatchMember *mem, const PairGroup *grp, BatchNow now, const int2 *ment, int nment,
                  int mon_from)
{
    extern __shared__ float lds[];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const bool mon = (int)blockIdx.x >= mon_from;
    int mi, sub = 0;
    PairGroup g = {-1, 0, 0};
    if (mon)
    {
        const int id = ((int)blockIdx.x - mon_from) * (NT / kWave) + wave;
        if (id >= nment)
            return;
        const int2 e = ment[id];
        mi = e.x;
        sub = e.y;
    }
    else
    {
        g = grp[blockIdx.x];
        mi = g.mem;
    }
    if (mi < 0)
        return;
    const BatchMember &m = mem[mi];
    const BatchClock t = now();
    const int n = member_step(m, t);
    if (n + 1 >= m.nend)
        return;
    PairArgs a = m.pa;
    const int s = member_buf(m, n, t), vs = member_vs(m, t);
    a.A = m.buf[s];
    a.B = m.buf[s ^ 1];
    a.Vs = m.vs[vs];
    a.Vs2 = m.vs[vs ^ 1];
    a.fold.sv = m.sv[n];
    a.sv1 = m.sv[n + 1];
    if (mon)
    {
        MonitorArgs o = {};
        o.pv = member_view(m, n, t);
        o.pv.fold = a.fold;
        o.n = n;
        o.np = m.np;
        o.pcells = m.pcells;
        o.poff = m.poff;
        o.ppol = m.ppol;
        o.ploop = m.ploop;
        o.prec = m.prec;
        o.npr = m.npr;
        o.prcell = m.prcell;
        o.inv_dl = m.inv_dl;
        o.prrec = m.prrec;
        monitor_pair(o, a, sub);
        return;
    }
    pair_tile<STUBS, false, C, NT>(a, g.tz, g.tt, (a.tb + 2 * a.hb) / C, lds);
}

// Per-slab maxima of the 16-bit members (one workgroup per (member, slab)).
static __global__ void k_slab_max_batch(const BatchMember *mem, const int2 *ent, BatchNow now)
{
    const int2 e = ent[blockIdx.x];
    const BatchMember &m = mem[e.x];
    const int n = member_step(m, now());
    if (n >= m.nend)
        return;
    __shared__ float s[256];
    const float *row = m.st.mpart + (size_t)e.y * m.st.strips;
    float v = 0.f;
    for (int t = threadIdx.x; t < m.st.strips; t += blockDim.x)
        v = fmaxf(v, row[t]);
    s[threadIdx.x] = v;
    __syncthreads();
    for (int w = blockDim.x / 2; w > 0; w >>= 1)
    {
        if ((int)threadIdx.x < w)
            s[threadIdx.x] = fmaxf(s[threadIdx.x], s[threadIdx.x + w]);
        __syncthreads();
    }
    if (threadIdx.x == 0)
        m.mreg[e.y] = s[0];
}

// Advances the clock.
static __global__ void k_tick(BatchClock *now, BatchClock by)
{
    if (threadIdx.x == 0 && blockIdx.x == 0)
    {
        now->tick += by.tick;
        now->launch += by.launch;
        now->pair += by.pair;
    }
}

} // namespace tlm
