// tlm_step2.h - two time steps of an FP32 grid in one pass over memory.
//
// k_step reads and writes every pulse once a step, which bounds a large grid
// by HBM bandwidth (12 + 12 floats per cell and step). k_step2 takes a pair
// of steps n, n+1. A workgroup owns a tile of consecutive 64-cell blocks of a
// slab and marches it along z: it scatters step n in the tile and in a rim of
// one row (nx cells) on either side, exchanges the reflected pulses (x and y
// faces through LDS, z faces in registers from slab to slab) and scatters step n+1 in the tile one slab behind. The rim's step n is
// computed again by the neighbouring tile, so no tile waits for another. Each
// cell's arithmetic is that of two k_step launches, in the same order, so the
// pulses, stubs and records are the same bits.
//
// What bounds it: HBM on large grids, now at 107 algorithmic bytes per cell
// for two steps instead of for one (512^3 free space: 7.35 GB fetched and
// 6.45 GB written a pair, 5.2 TB/s, against 13.0 GB at 5.9 TB/s for one
// k_step); the launch and the loads' latency on small ones. us a step, two
// k_step launches against a pair: 512^3 64 boxes 2520 / 1380 to 1530 from box
// to box, free space 2180 / 1320, 256^3 8 boxes 285 / 171, 128^3 33.4 / 21.2,
// 64^3 7.9 / 5.5, 24^3 4.8 / 3.0.
// Tried and not kept: x pulses exchanged between lanes instead of through LDS
// (512^3 free space 1.35 against 1.33 ms, 64^3 6.0 against 4.7 us), x by y
// tiles with a rim on all four sides (the rim's columns cost whole lines:
// 512^3 64 boxes 1.67 to 2.4 ms), non-temporal stores (1.35 against 1.33 ms)
// and loads (1.75: a tile's rim is found in L2 only if it stays there), three
// and four blocks per wave (1.62, 1.69 ms), more waves at fewer registers
// (spills: 2.9 ms and up).
//
// A tile is a run of whole blocks, whatever nx is, so every load and store of
// a wave is one aligned 256-byte run per port (but for the y faces it pushes
// where nx is no multiple of 64).
//
// Stubs are read from Vs and written to Vs2 (a rim cell's stubs are read by
// a tile that does not own them, so the pair cannot update them in place).
// The intermediate pulses never reach memory; the monitors of step n+1
// recompute them for the cells they need (PairPulses), seven cells' work for
// each, so contexts with very many records keep single steps (pair_suits).
#pragma once

#include "tlm_kernels.h"

namespace tlm {

struct PairArgs
{
    const char *A;        // incident pulses of step n
    char *B;              // incident pulses of step n+2
    const float *Vs;      // stubs before step n
    float *Vs2;           // stubs after step n+1
    const uint16_t *code;
    const uint8_t *uair;  // block flags (StepArgs::uair)
    const float4 *props;
    double *epart;        // energy partials of step n, one per 64-cell block
    int nx, ny, nz;
    long long Pp;         // slab pitch (cells)
    float rho;
    int nmat;
    int strips;           // 64-cell blocks per slab
    int tb, hb;           // blocks of a tile and of its rim on either side
    int ntile;            // tiles per slab
    int zc;               // slabs per tile
    XcdMap xm;            // workgroup -> tile
    Magic mPp, mnx;       // division by the slab pitch and by nx
    Fold fold;            // soft sources of step n (fold.sv) ...
    float sv1;            // ... and the waveform value of step n+1
};

// Lane facts of a tile cell, in one word.
enum : unsigned
{
    TF_ACT = 1u, // a grid cell of the tile
    TF_X0 = 2u,  // outer faces
    TF_X1 = 4u,
    TF_Y0 = 8u,
    TF_Y1 = 16u
};

// Byte offset of in-slab cell g's first stub inside its slab.
__device__ __forceinline__ unsigned stub_off(unsigned g)
{
    return (g >> 6) * 768u + (g & 63u) * 4u;
}

// One step-n scatter of a loaded cell: o = reflected pulses (a PEC cell keeps
// its incident ones), st updated.
template <bool STUBS>
__device__ __forceinline__ void pair_scatter(const float v[12], unsigned code, float st[3],
                                             const float2 *tab, float o[12])
{
    const unsigned m = code & 0xFFu;
    if (STUBS && m >= 2u)
    {
        const float2 pr = tab[m - 2u];
        scn::scatter_diel(v, st, pr.x, pr.y, o);
    }
    else
        scn::scatter_air(v, o);
    if (__any(m == 1u))
    {
#pragma unroll
        for (int p = 0; p < 12; ++p)
            o[p] = m == 1u ? v[p] : o[p];
    }
}

// ---- monitors of steps n and n+1 ------------------------------------------
// The incident pulses of cell c at step n+1, from A. Eight lanes take one
// cell: lane q scatters the neighbour across face q (0..5: x-, x+, y-, y+,
// z-, z+) or the cell itself (6, 7), so the loads of all seven cells are in
// flight together, and the group exchanges the pulses by shuffles. w: the
// pulses of step n+1 (every lane); v: the lane's own gather, in lanes 6 and 7
// the cell's pulses of step n.
struct PairPulses
{
    const PulseView &pv; // pulses and folded sources of step n
    const PairArgs &a;

    __device__ __forceinline__ void operator()(long long c, float v[12], float w[12]) const
    {
        const int q = threadIdx.x & 7;
        const int k = (int)mdiv((unsigned)c, a.mPp);
        const int f = (int)(c - (long long)k * a.Pp);
        const int j = (int)mdiv((unsigned)f, a.mnx), i = f - j * a.nx;
        const unsigned code0 = a.code[c];
        const bool pec = (code0 & 0xFFu) == 1u;
        const int ax = q >> 1, hi = q & 1;
        const int co = ax == 0 ? i : ax == 1 ? j : k, nn = ax == 0 ? a.nx : ax == 1 ? a.ny : a.nz;
        const bool self = q >= 6 || (hi ? co == nn - 1 : co == 0);
        const long long stride = ax == 0 ? 1 : ax == 1 ? a.nx : a.Pp;
        const long long d = self ? c : c + (hi ? stride : -stride);
        const unsigned cd = a.code[d], m = cd & 0xFFu;
        float o[12], st[3];
        pv_get12<PF_F32>(pv, d, v);
        if (cd & kCodeSource)
            fold_sources(a.fold, d, v);
        __builtin_amdgcn_sched_barrier(0);
        if (m >= 2u)
        {
            const float *S = a.Vs + (size_t)(d >> 6) * kStubBlock + (d & (kWave - 1));
            const float4 pr = a.props[m - 2u];
#pragma unroll
            for (int s = 0; s < 3; ++s)
                st[s] = S[s * kWave];
            scn::scatter_diel(v, st, pr.x, pr.z, o);
        }
        else
            scn::scatter_air(v, o);
        if (m == 1u)
        {
#pragma unroll
            for (int p = 0; p < 12; ++p)
                o[p] = v[p];
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int s = 0; s < 6; ++s)
        {
            const int sa = s >> 1, sh = s & 1;
            const int sc = sa == 0 ? i : sa == 1 ? j : k, sn = sa == 0 ? a.nx : sa == 1 ? a.ny : a.nz;
            const bool bnd = sh ? sc == sn - 1 : sc == 0;
            const bool pecN = (code0 & (NB_XM << s)) != 0u;
            // the opposite face of the neighbour, scattered by lane s
            const int opp = 4 * sa + (sh ? 0 : 2);
            const float n0 = __shfl(o[opp], s, 8), n1 = __shfl(o[opp + 1], s, 8);
            const float o0 = __shfl(o[2 * s], 6, 8), o1 = __shfl(o[2 * s + 1], 6, 8);
            w[2 * s] = bnd ? a.rho * o0 : pec ? o0 : pecN ? -o0 : n0;
            w[2 * s + 1] = bnd ? a.rho * o1 : pec ? o1 : pecN ? -o1 : n1;
        }
        if (code0 & kCodeSource)
        {
            Fold fn = a.fold;
            fn.sv = a.sv1;
            fold_sources(fn, c, w);
        }
    }
};

// Waves that take the records of a pair: eight faces or probes to a wave
// (eight lanes each), then one wave for each port.
__host__ __device__ inline int pair_face_waves(const MonitorArgs &m)
{
    return (m.nf + m.nh + m.npr + 7) / 8;
}
// Records of steps n and n+1 by wave `wave` of them; lane 6 of a group writes.
__device__ __forceinline__ void monitor_pair(const MonitorArgs &m, const PairArgs &a, int wave)
{
    const PairPulses at{m.pv, a};
    const int lane = threadIdx.x & (kWave - 1), grp = lane >> 3;
    const int n = m.n;
    const int fw = pair_face_waves(m);
    const bool port = wave >= fw;
    int id = port ? wave - fw : wave * 8 + grp;
    if (port ? id >= m.np : id >= m.nf + m.nh + m.npr)
        return;
    // entries of a port: its cells, then the four cells of the current loop
    const int b = port ? m.poff[id] : 0, nc = port ? m.poff[id + 1] - b : 1;
    const int ne = port ? (nc > 0 ? nc + 4 : 0) : 1;
    const int pol = port ? m.ppol[id] : 0, t1 = (pol + 1) % 3, t2 = (pol + 2) % 3;
    const int kind = id < m.nf ? 0 : id < m.nf + m.nh ? 1 : 2;
    const int sub = kind == 0 ? id : kind == 1 ? id - m.nf : id - m.nf - m.nh;
    float vs0 = 0.f, vs1 = 0.f, z0 = 0.f, z1 = 0.f;
    for (int s0 = 0; s0 < ne; s0 += 8)
    {
        const int s = port ? min(s0 + grp, ne - 1) : 0;
        const long long c = port ? (s < nc ? m.pcells[b + s] : m.ploop[4 * (size_t)id + (s - nc)])
                            : kind == 0 ? m.fcell[sub]
                            : kind == 1 ? m.hcell[sub]
                                        : m.prcell[sub];
        float v[12], w[12];
        at(c, v, w);
        if (port)
        {
            // V_j of a port cell, or the loop's circulation, added in list order
            const int ax = s - nc < 2 ? t2 : t1;
            const float x = s < nc ? scn::vj(v, pol) : scn::zi(v, ax);
            const float y = s < nc ? scn::vj(w, pol) : scn::zi(w, ax);
            for (int g = 0; g < 8 && s0 + g < ne; ++g)
            {
                const float p = __shfl(x, g * 8 + 6), q = __shfl(y, g * 8 + 6);
                const int e = s0 + g - nc;
                if (e < 0)
                {
                    vs0 += p;
                    vs1 += q;
                }
                else if (e == 0 || e == 3)
                {
                    z0 += p;
                    z1 += q;
                }
                else
                {
                    z0 -= p;
                    z1 -= q;
                }
            }
        }
        else if ((lane & 7) == 6)
        {
            if (kind == 0)
            {
                js_record(m, sub, n, v);
                js_record(m, sub, n + 1, w);
            }
            else if (kind == 1)
            {
                if (n >= m.settle)
                    huy_record(m, sub, n, v);
                if (n + 1 >= m.settle)
                    huy_record(m, sub, n + 1, w);
            }
            else
            {
                probe_record(v, sub, n, m.npr, m.inv_dl, m.prrec);
                probe_record(w, sub, n + 1, m.npr, m.inv_dl, m.prrec);
            }
        }
    }
    if (port && lane == 0)
    {
        const bool any = nc > 0;
        port_record(vs0, any ? -2.0f * z0 / ETA0 : 0.f, id, n, m.np, m.prec);
        port_record(vs1, any ? -2.0f * z1 / ETA0 : 0.f, id, n + 1, m.np, m.prec);
    }
}

// Barrier for data exchanged through LDS only: global loads and stores stay
// in flight across it.
__device__ __forceinline__ void pair_barrier()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Waves per SIMD that the registers leave room for: 128 VGPRs, in which both
// variants of two blocks per wave fit without spills. One workgroup of 16 waves fills a CU.
constexpr int kPairOcc = 4;

// ---- the pair -------------------------------------------------------------
// LDS bytes: the x and y pulses of two slabs and the material table.
template <int C, int NT> constexpr int pair_lds(int nmat)
{
    return 2 * C * NT * 32 + nmat * 8;
}

// Tile tt of the slabs' tiles from slab tz * zc on, by the workgroup's first
// nw waves (tb + 2 hb blocks, C to a wave).
template <bool STUBS, bool ENERGY, int C, int NT>
__device__ __forceinline__ void pair_tile(const PairArgs &a, int tz, int tt, int nw, float *lds)
{
    const int nt = (int)blockDim.x;
    constexpr int em = C * NT;
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int b0 = tt * a.tb, b1 = min(a.strips, b0 + a.tb); // blocks of the tile
    const int k0 = tz * a.zc, k1 = min(a.nz, k0 + a.zc);
    const int ka = max(0, k0 - 1), klast = min(k1, a.nz - 1); // slabs read
    const int nxy = a.nx * a.ny;
    const float rho = a.rho;
    const size_t slabB = (size_t)a.Pp * 48u;
    float *const X = lds; // [2][8][em]: reflected x and y pulses (ports 0..7) of two slabs
    float2 *const tab = reinterpret_cast<float2 *>(lds + 16 * em);
    if (STUBS)
    {
        for (int q = threadIdx.x; q < a.nmat; q += nt)
        {
            const float4 pr = a.props[q];
            tab[q] = make_float2(pr.x, pr.z);
        }
        __syncthreads();
    }
    if (wave >= nw)
        return;

    // A wave holds C blocks, all of the tile (waves below ni) or all of the rim.
    const int ni = a.tb / C;
    const bool rim = wave >= ni;
    int f[C], bi[C]; // cell inside the slab (clamped into the cells read), block inside the tile and rim
    unsigned tf[C];
    float v[C][12], s[C][3]; // pulses, stubs and code of the slab, loaded one slab ahead
    unsigned code[C];
#pragma unroll
    for (int c = 0; c < C; ++c)
    {
        // places past the tile's or the rim's last block take that block again
        // (the same values in the same slots)
        if (!rim)
            bi[c] = a.hb + min(c * ni + wave, b1 - b0 - 1);
        else
        {
            const int r = min(c * (nw - ni) + wave - ni, 2 * a.hb - 1);
            bi[c] = r < a.hb ? r : r + (b1 - b0);
        }
        const int g = (b0 - a.hb + bi[c]) * kWave + lane; // the lane's cell; past the rim, one of the rim's
        f[c] = min(max(g, max(0, b0 * kWave - a.nx)), min(nxy, b1 * kWave + a.nx) - 1);
        const int j = (int)mdiv((unsigned)f[c], a.mnx), i = f[c] - j * a.nx;
        const bool act = !rim && g < nxy;
        tf[c] = (act ? TF_ACT : 0u) | (i == 0 ? TF_X0 : 0u) | (i == a.nx - 1 ? TF_X1 : 0u) |
                (j == 0 ? TF_Y0 : 0u) | (j == a.ny - 1 ? TF_Y1 : 0u);
#pragma unroll
        for (int p = 0; p < 3; ++p)
            s[c][p] = 0.f;
    }
    // The loads of a slab are issued one slab ahead, right after the registers'
    // last use; none is skipped (lanes with nothing to load repeat a cell of
    // the rim), so that the number of loads and stores in flight behind them
    // is known and a wait for them leaves the stores issued later in flight.
    auto load = [&](int kk, int c) {
        const int k = min(kk, klast);
        const char *Ak = a.A + (size_t)k * slabB;
        const unsigned off = blk_off((unsigned)f[c]);
        if (STUBS)
        {
            // block flag bits 3 and 4: a dielectric cell among the block's cells 0-31 / 32-63
            const int g = min(max(b0 - a.hb + __builtin_amdgcn_readfirstlane(bi[c]), 0), a.strips - 1);
            const unsigned fl = block_flag(a.uair, (size_t)k * a.strips + g);
            if ((fl >> (3 + (lane >> 5))) & 1u)
            {
                const char *S = reinterpret_cast<const char *>(a.Vs + (size_t)k * a.strips * kStubBlock);
                const unsigned so = stub_off((unsigned)f[c]);
#pragma unroll
                for (int p = 0; p < 3; ++p)
                    s[c][p] = ldo(S + p * 256, so);
            }
        }
        code[c] = ldc(a.code + (size_t)k * a.Pp, (unsigned)f[c]);
#pragma unroll
        for (int p = 0; p < 12; ++p)
            v[c][p] = ldo(Ak + p * 256, off);
    };
    // Step n of block c of slab kk: reflected pulses o, stubs sn; the pulses
    // the neighbouring blocks need go to LDS.
    auto scatter1 = [&](int kk, int c, float o[12], float sn[3]) {
        const int e = bi[c] * kWave + lane;
#pragma unroll
        for (int p = 0; p < 3; ++p)
            sn[p] = s[c][p];
        if (code[c] & kCodeSource)
            fold_sources(a.fold, (long long)kk * a.Pp + f[c], v[c]);
        const bool in = kk >= k0 && kk < k1;
        if (ENERGY && in && !rim) // a place past the last block stores that block's sum again
            block_energy((tf[c] & TF_ACT) ? cell_energy(v[c]) : 0.0, lane,
                         a.epart + (size_t)kk * a.strips + (b0 - a.hb + bi[c]));
        pair_scatter<STUBS>(v[c], code[c], sn, tab, o);
        if (in)
        {
            float *const Xw = X + (kk & 1) * (8 * em) + e;
#pragma unroll
            for (int p = 0; p < 8; ++p)
                Xw[p * em] = o[p];
        }
    };

    if (rim)
    {
        // the rim's waves scatter step n of the tile's slabs and keep the
        // tile's barriers
#pragma unroll
        for (int c = 0; c < C; ++c)
            load(k0, c);
        for (int kk = ka; kk <= k1; ++kk)
        {
            if (kk >= k0 && kk < k1)
            {
#pragma unroll
                for (int c = 0; c < C; ++c)
                {
                    __builtin_amdgcn_sched_barrier(0);
                    float o[12], sn[3];
                    scatter1(kk, c, o, sn);
                    load(kk + 1, c);
                }
            }
            pair_barrier();
        }
        return;
    }

    unsigned cd[C];
    float h8[C], h9[C], zu0[C], zu1[C], st[C][3]; // the slab before: incident z- pulses, z+ sent, stubs
#pragma unroll
    for (int c = 0; c < C; ++c)
    {
        zu0[c] = zu1[c] = 0.f;
        load(ka, c);
    }
    // What step n+1 of slab kk takes from the slab below.
    auto keep = [&](int kk, int c, unsigned q1, const float o[12], const float sn[3]) {
        const bool pec = (q1 & 0xFFu) == 1u, pz = (q1 & NB_ZM) != 0u;
        h8[c] = kk == 0 ? rho * o[8] : pec ? o[8] : pz ? -o[8] : zu0[c];
        h9[c] = kk == 0 ? rho * o[9] : pec ? o[9] : pz ? -o[9] : zu1[c];
        zu0[c] = o[10];
        zu1[c] = o[11];
        cd[c] = q1;
#pragma unroll
        for (int p = 0; p < 3; ++p)
            st[c][p] = sn[p];
    };
    // the slabs before the first that can be finished
    for (int kk = ka; kk <= k0; ++kk)
    {
#pragma unroll
        for (int c = 0; c < C; ++c)
        {
            float o[12], sn[3];
            scatter1(kk, c, o, sn);
            const unsigned q1 = code[c];
            load(kk + 1, c);
            keep(kk, c, q1, o, sn);
        }
        pair_barrier();
    }
    for (int kk = k0 + 1; kk <= k1; ++kk)
    {
        const int kp = kk - 1;
        const float *const Xr = X + (kp & 1) * (8 * em);
        char *const Bk = a.B + (size_t)kp * slabB;
#pragma unroll
        for (int c = 0; c < C; ++c)
        {
            // one block after the other: interleaved, they would need more registers
            __builtin_amdgcn_sched_barrier(0);
            // what follows from the cell's place is computed anew for each slab:
            // held across the march, it would not fit the registers
            asm volatile("" : "+v"(f[c]), "+v"(tf[c]));
            const int e = bi[c] * kWave + lane;
            const unsigned t = tf[c];
            float o[12], sn[3];
            scatter1(kk, c, o, sn); // past the grid: a slab again, not used
            const unsigned q1 = code[c];
            load(kk + 1, c);

            // step n+1 of slab kp
            const unsigned q = cd[c];
            const bool pec = (q & 0xFFu) == 1u;
            // no PEC cell, PEC neighbour, outer face, source or padding in the wave
            const bool plain = kp > 0 && kp < a.nz - 1 && !__any((q & 0xFFu) == 1u || (q & 0x7F00u) != 0u || t != TF_ACT);
            float in2[12], o2[12];
            in2[8] = h8[c];
            in2[9] = h9[c];
            const unsigned fu = (unsigned)f[c];
            const unsigned off = (unsigned)(b0 - a.hb + bi[c]) * 3072u + (unsigned)lane * 4u;
            if (plain)
            {
                in2[0] = Xr[2 * em + e - 1];
                in2[1] = Xr[3 * em + e - 1];
                in2[2] = Xr[0 * em + e + 1];
                in2[3] = Xr[1 * em + e + 1];
                in2[4] = Xr[6 * em + e - a.nx];
                in2[5] = Xr[7 * em + e - a.nx];
                in2[6] = Xr[4 * em + e + a.nx];
                in2[7] = Xr[5 * em + e + a.nx];
                in2[10] = o[8];
                in2[11] = o[9];
            }
            else
            {
                // the neighbour's pulse, or the cell's own where the link is broken
                auto take = [&](int p, int opp, int nbe, unsigned bbit, unsigned pbit) {
                    const bool bnd = (t & bbit) != 0u, pecN = (q & pbit) != 0u;
                    const bool mine = pec || bnd || pecN || !(t & TF_ACT);
                    const float sc = bnd ? rho : (pecN && !pec) ? -1.0f : 1.0f;
                    const int ad = mine ? p * em + e : opp * em + nbe;
                    in2[p] = sc * Xr[ad];
                    in2[p + 1] = sc * Xr[ad + em];
                };
                take(0, 2, e - 1, TF_X0, NB_XM);
                take(2, 0, e + 1, TF_X1, NB_XP);
                take(4, 6, e - a.nx, TF_Y0, NB_YM);
                take(6, 4, e + a.nx, TF_Y1, NB_YP);
                const bool top = kp == a.nz - 1, pz = (q & NB_ZP) != 0u;
                in2[10] = top ? rho * zu0[c] : pec ? zu0[c] : pz ? -zu0[c] : o[8];
                in2[11] = top ? rho * zu1[c] : pec ? zu1[c] : pz ? -zu1[c] : o[9];
                if (q & kCodeSource)
                {
                    Fold fn = a.fold;
                    fn.sv = a.sv1;
                    fold_sources(fn, (long long)kp * a.Pp + f[c], in2);
                }
            }
            pair_scatter<STUBS>(in2, q, st[c], tab, o2);
            if (STUBS)
            {
                const unsigned fl = block_flag(a.uair, (size_t)kp * a.strips + b0 - a.hb + __builtin_amdgcn_readfirstlane(bi[c]));
                if (((fl >> (3 + (lane >> 5))) & 1u) && (t & TF_ACT))
                {
                    char *S = reinterpret_cast<char *>(a.Vs2 + (size_t)kp * a.strips * kStubBlock);
                    const unsigned so = stub_off(fu);
#pragma unroll
                    for (int p = 0; p < 3; ++p)
                        sto<false>(S + p * 256, so, st[c][p]);
                }
            }
            // Every pulse is pushed into the neighbour's slot; where the link is
            // broken the cell keeps it. Lanes past the grid fill their own slots
            // of the slab's padding, which nothing reads: no store is skipped.
            if (plain)
            {
                const unsigned aL = blk_off(fu - 1u), aR = blk_off(fu + 1u);
                sto<false>(Bk + 2 * 256, aL, o2[0]);
                sto<false>(Bk + 3 * 256, aL, o2[1]);
                sto<false>(Bk, aR, o2[2]);
                sto<false>(Bk + 256, aR, o2[3]);
                const unsigned aM = blk_off(fu - (unsigned)a.nx), aP = blk_off(fu + (unsigned)a.nx);
                sto<false>(Bk + 6 * 256, aM, o2[4]);
                sto<false>(Bk + 7 * 256, aM, o2[5]);
                sto<false>(Bk + 4 * 256, aP, o2[6]);
                sto<false>(Bk + 5 * 256, aP, o2[7]);
                sto<false>(Bk - slabB + 10 * 256, off, o2[8]);
                sto<false>(Bk - slabB + 11 * 256, off, o2[9]);
                sto<false>(Bk + slabB + 8 * 256, off, o2[10]);
                sto<false>(Bk + slabB + 9 * 256, off, o2[11]);
            }
            else
            {
                const bool idle = !(t & TF_ACT);
                auto give = [&](int p, int opp, unsigned nboff, unsigned bbit, unsigned pbit) {
                    const bool bnd = (t & bbit) != 0u, pecN = (q & pbit) != 0u;
                    const bool mine = pec || bnd || pecN || idle;
                    const float sc = bnd ? rho : (pecN && !pec) ? -1.0f : 1.0f;
                    const unsigned ad = mine ? off + p * 256u : nboff + opp * 256u;
                    sto<false>(Bk, ad, sc * o2[p]);
                    sto<false>(Bk + 256, ad, sc * o2[p + 1]);
                };
                give(0, 2, blk_off(fu - 1u), TF_X0, NB_XM);
                give(2, 0, blk_off(fu + 1u), TF_X1, NB_XP);
                give(4, 6, blk_off(fu - (unsigned)a.nx), TF_Y0, NB_YM);
                give(6, 4, blk_off(fu + (unsigned)a.nx), TF_Y1, NB_YP);
                auto give_z = [&](int p, int opp, bool bnd, bool pecN, char *Bn) {
                    const bool mine = pec || bnd || pecN || idle;
                    const float sc = bnd ? rho : (pecN && !pec) ? -1.0f : 1.0f;
                    char *const w = (mine ? Bk + p * 256 : Bn + opp * 256) + off;
                    *reinterpret_cast<float *>(w) = sc * o2[p];
                    *reinterpret_cast<float *>(w + 256) = sc * o2[p + 1];
                };
                give_z(8, 10, kp == 0, (q & NB_ZM) != 0u, Bk - slabB);
                give_z(10, 8, kp == a.nz - 1, (q & NB_ZP) != 0u, Bk + slabB);
            }
            keep(kk, c, q1, o, sn);
        }
        pair_barrier();
    }
}

template <bool STUBS, bool ENERGY, int C, int NT>
__global__ void __launch_bounds__(NT, kPairOcc) k_step2(PairArgs a, MonitorArgs m, int mon_from, int mon_plane)
{
    extern __shared__ float lds[];
    const int nt = (int)blockDim.x, nw = nt / kWave;
    if ((int)blockIdx.x >= mon_from)
    {
        // the faces, probes and ports of both steps, then the plane of step n
        const int b = (int)blockIdx.x - mon_from;
        if (b < mon_plane)
            monitor_pair(m, a, (b * nt + (int)threadIdx.x) / kWave);
        else if ((b - mon_plane) * nt + (int)threadIdx.x < m.pn)
            plane_item<PF_F32>(m, (b - mon_plane) * nt + (int)threadIdx.x);
        return;
    }
    const XcdRange gr = xcd_range_map(blockIdx.x, a.xm);
    if (gr.first >= gr.end)
        return;
    const int tz = gr.first / a.ntile;
    pair_tile<STUBS, ENERGY, C, NT>(a, tz, gr.first - tz * a.ntile, nw, lds);
}

} // namespace tlm
