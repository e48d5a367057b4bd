// TlmFarField.hip - near-to-far-field transform from the Huygens box DFTs
// on the device (ComputeFarFieldFromHuygens, TlmSolver.cpp:805-916).
//
// The reference evaluates, for every (theta, phi) of the output grid, a
// float sum over all Huygens faces of the face's equivalent currents times
// exp(+j k0 r.r'), on the host thread pool: O(directions x faces) sin/cos.
// Here, two ways to the vector sums S_J = sum J e^{j phase} and S_M per
// direction (J' = n x (eta0 H), M = -(n x E) in world components,
// TlmSolver.cpp:823-843):
//   any faces    k_ff_faces_* make one record per face (position, currents),
//                k_ff_sums takes some directions and a range of faces per
//                workgroup, a phase factor per face and pair of opposite directions;
//   a context's  the faces of a Huygens box lie on the lattice of cell
//   box          centres, so the phase factor is a product over the axes:
//                per direction and plane, sum_v E_v sum_u E_u J(u, v). k_ff_phase
//                tabulates the factors of each axis, k_ff_lattice does the
//                inner sums as a matrix product on the FP32 matrix cores
//                (directions x u times u x (v, current)).
// k_ff_finish adds the partial sums in double in a fixed order, projects on
// theta-hat / phi-hat (N_theta = S_J . theta-hat etc.) and takes
// U = |L_phi + N_theta|^2 + |L_theta - N_phi|^2.
// Phases are reduced to a fraction of a turn in double: a box of 250 cells is
// some 70 rad from side to side, where float phases are off by 4e-6. The norm
// of U's error against sums in 64 bits, 1.2e-6 with those, is 9e-8.
// The projections are taken after the sum instead of per face (the same linear
// map), so U agrees with the reference's float sums to their rounding, not bit
// for bit. The directivity and peak search run on the host over U exactly as
// TlmSolver.cpp:893-913.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Wunused-function" // the step kernels of the shared header
#include "tlm_context.h"
#pragma clang diagnostic pop

#include <hip/hip_runtime.h>

#include <cmath>
#include <cstring>
#include <mutex>
#include <string>
#include <vector>

using namespace tlmi;

namespace {

constexpr int kFfThreads = 256;
constexpr int kSums = 8;  // vector sums per thread of k_ff_sums
constexpr int kAcc = 12;  // S_J (re x,y,z; im x,y,z), S_M (same)
constexpr int kTile = 32; // directions per workgroup of k_ff_lattice
constexpr int kOut = 32;  // directions per workgroup of k_ff_finish
constexpr double kC0 = 299792458.0;

// The output grid: ang[0, nT) = (cos, sin) of theta, ang[nT, nT + nP) of phi;
// kt = 1 / wavelength, turns per metre.
// Opposite directions have conjugate phase factors, so that one set of
// products gives the sums of both. With nP odd the grid holds the opposite of
// each of its directions, (pi - theta, phi + pi), and phi = 2 pi is phi = 0
// again: the sums are taken over h = (nP - 1) / 2 values of phi, for each
// direction e and (o = 1) its opposite. Else (h = 0) over the whole grid.
struct FfDirs
{
    const double2 *ang;
    int nT, nP, h;
    double kt;
    __host__ __device__ int n() const
    {
        return nT * (h ? h : nP);
    }
    __host__ __device__ int sides() const
    {
        return h ? 2 : 1;
    }
    // theta and phi index of sum e, side o
    __device__ int2 at(int e, int o) const
    {
        const int w = h ? h : nP, t = e / w, p = e - t * w;
        return o ? make_int2(nT - 1 - t, p + h) : make_int2(t, p);
    }
    // component q of the wave vector, in turns per metre
    __device__ double wave(int e, int q) const
    {
        const int2 g = at(e, 0);
        const double2 t = ang[g.x], p = ang[nT + g.y];
        return kt * (q == 0 ? t.y * p.x : q == 1 ? t.y * p.y : t.x);
    }
};

// Partial sums: part[((range * kAcc + q) * sides + o) * pitch + e].

// Face record: px py pz pad | jr(3) ji(3) | mr(3) mi(3)
struct FfFace
{
    float4 a, b, c, d;
};

__device__ __constant__ int kTan[3][2] = {{1, 2}, {0, 2}, {0, 1}}; // POL, TlmSolver.cpp:23

// Currents of one face from its 8 DFT floats (E1, E2, eta0 H1, eta0 H2 as
// re, im), axis and outward sign (TlmSolver.cpp:823-843).
__device__ FfFace make_face(float px, float py, float pz, int ax, float s, const float *a)
{
    const int t1 = kTan[ax][0], t2 = kTan[ax][1];
    const float sa = (ax == 1) ? -1.0f : 1.0f;
    float jr[3] = {0.f, 0.f, 0.f}, ji[3] = {0.f, 0.f, 0.f};
    float mr[3] = {0.f, 0.f, 0.f}, mi[3] = {0.f, 0.f, 0.f};
    jr[t2] = s * sa * a[4];
    ji[t2] = s * sa * a[5];
    jr[t1] = -s * sa * a[6];
    ji[t1] = -s * sa * a[7];
    mr[t2] = -s * sa * a[0];
    mi[t2] = -s * sa * a[1];
    mr[t1] = s * sa * a[2];
    mi[t1] = s * sa * a[3];
    FfFace f;
    f.a = make_float4(px, py, pz, 0.f);
    f.b = make_float4(jr[0], jr[1], jr[2], ji[0]);
    f.c = make_float4(ji[1], ji[2], mr[0], mr[1]);
    f.d = make_float4(mr[2], mi[0], mi[1], mi[2]);
    return f;
}

// Faces given by the caller: positions, sides (axis, and 4 if the outward
// sign is negative).
__global__ void k_ff_faces_host(int nf, const float *pos, const uint8_t *side, const float *dft,
                                FfFace *out)
{
    const int f = blockIdx.x * blockDim.x + threadIdx.x;
    if (f >= nf)
        return;
    out[f] = make_face(pos[3 * f], pos[3 * f + 1], pos[3 * f + 2], side[f] & 3, side[f] & 4 ? -1.f : 1.f,
                       dft + 8 * (long long)f);
}

// Faces of a context: padded cells, axes and the resident accumulators.
__global__ void k_ff_faces_ctx(int nf, const long long *pcell, const int *axis, const float *dft,
                               int nx, int ny, int nz, long long Pp, float ox, float oy, float oz,
                               float dl, FfFace *out)
{
    const int f = blockIdx.x * blockDim.x + threadIdx.x;
    if (f >= nf)
        return;
    const long long p = pcell[f];
    const long long k = p / Pp;
    const long long r = p - k * Pp;
    const int j = (int)(r / nx);
    const int i = (int)(r - (long long)j * nx);
    // HuyFace::pos = cellCenter - (origin + (n dl) * 0.5) (TlmSolver.cpp:323, 334)
    const float cx = ox + (nx * dl) * 0.5f, cy = oy + (ny * dl) * 0.5f, cz = oz + (nz * dl) * 0.5f;
    const float px = (ox + (i + 0.5f) * dl) - cx;
    const float py = (oy + (j + 0.5f) * dl) - cy;
    const float pz = (oz + ((int)k + 0.5f) * dl) - cz;
    const int a = axis[f];
    const int co = a == 0 ? i : (a == 1 ? j : (int)k);
    const int nn = a == 0 ? nx : (a == 1 ? ny : nz);
    const float s = (2 * co + 1 < nn) ? -1.0f : 1.0f; // low side of the box: outward -e_a
    out[f] = make_face(px, py, pz, a, s, dft + 8 * (long long)f);
}

// Sums over the wave of 96 values per lane: in each of five steps a lane
// passes half of its values to its partner and adds the partner's to the half
// it keeps, which takes 96 exchanges where a full reduction of each takes 576.
// v[0..2] are then the sums of values first..first + 2 (returned), alike in
// pairs of lanes.
__device__ inline int wave_sums(float (&v)[96])
{
    int first = 0;
#pragma unroll
    for (int h = 48, o = 32; h >= 3; h /= 2, o /= 2)
    {
        const bool up = threadIdx.x & o;
        first += up ? h : 0;
#pragma unroll
        for (int i = 0; i < h; ++i)
        {
            const float give = up ? v[i] : v[i + h], keep = up ? v[i + h] : v[i];
            v[i] = keep + __shfl_xor(give, o, 64);
        }
    }
#pragma unroll
    for (int i = 0; i < 3; ++i)
        v[i] += __shfl_xor(v[i], 1, 64);
    return first;
}

__device__ inline double uniform(double x)
{
    return __hiloint2double(__builtin_amdgcn_readfirstlane(__double2hiint(x)),
                            __builtin_amdgcn_readfirstlane(__double2loint(x)));
}

// sin and cos of 2 pi t for |t| <= 1/2: t = q/2 + g with |g| <= 1/4, then
// sin(2 pi g) and cos(2 pi g) as polynomials in g^2 (interpolation at the
// Chebyshev nodes of [0, 1/16]; with float rounding 1.5e-7 and 1.1e-7 off at most).
__device__ __forceinline__ void sincos_turns(float t, float &s, float &c)
{
    const float q = __builtin_rintf(2.0f * t);
    const float g = __builtin_fmaf(q, -0.5f, t), x = g * g;
    float a = 39.759827f;
    a = __builtin_fmaf(a, x, -76.58117f);
    a = __builtin_fmaf(a, x, 81.60248f);
    a = __builtin_fmaf(a, x, -41.341682f);
    a = __builtin_fmaf(a, x, 6.2831855f);
    a *= g;
    float b = -24.981434f;
    b = __builtin_fmaf(b, x, 60.14389f);
    b = __builtin_fmaf(b, x, -85.45357f);
    b = __builtin_fmaf(b, x, 64.93935f);
    b = __builtin_fmaf(b, x, -19.739208f);
    b = __builtin_fmaf(b, x, 1.0f);
    s = q != 0.0f ? -a : a;
    c = q != 0.0f ? -b : b;
}

// Partial sums of faces [fr*per, min(nf, (fr+1)*per)) for the kSums / (1 +
// OPP) entries e of group blockIdx.x; OPP: and their opposites.
// Bound by VALU issue: per face and entry 6 operations of the phase (FP64, at
// FP32's rate here), 20 of the sine and cosine and 24 multiply-adds.
// 50021 faces x 37 x 73 directions: 353 us with sincosf, unfused products and
// each direction by itself, 182 with sincos_turns and multiply-adds, 149 with
// opposite directions together, 94 with wave_sums for 96 full reductions (of
// the 66 that its operations take).
template <bool OPP>
__global__ void __launch_bounds__(kFfThreads)
    k_ff_sums(const FfFace *faces, int nf, int per, FfDirs D, float *part)
{
    constexpr int kN = OPP ? kSums / 2 : kSums, kV = OPP ? 2 * kAcc : kAcc;
    __shared__ double rh[kN][3];
    __shared__ float wsum[kFfThreads / 64][kN * kV];
    const int e0 = blockIdx.x * kN, n = D.n();
    if (threadIdx.x < kN * 3)
    {
        const int d = threadIdx.x / 3, q = threadIdx.x % 3;
        rh[d][q] = e0 + d < n ? D.wave(e0 + d, q) : 0.0;
    }
    __syncthreads();
    // the same for all lanes: scalar registers, of which a wave has some to spare
    double k[kN][3];
#pragma unroll
    for (int d = 0; d < kN; ++d)
#pragma unroll
        for (int q = 0; q < 3; ++q)
            k[d][q] = uniform(rh[d][q]);
    float acc[kSums * kAcc]; // [entry][kV]
#pragma unroll
    for (int q = 0; q < kSums * kAcc; ++q)
        acc[q] = 0.f;
    const int fr = blockIdx.y;
    const int f1 = min(nf, (fr + 1) * per);
    for (int f = fr * per + threadIdx.x; f < f1; f += kFfThreads)
    {
        const FfFace F = faces[f];
        // J x, y, z, M x, y, z
        const float xr[6] = {F.b.x, F.b.y, F.b.z, F.c.z, F.c.w, F.d.x};
        const float xi[6] = {F.b.w, F.c.x, F.c.y, F.d.y, F.d.z, F.d.w};
        const double px = F.a.x, py = F.a.y, pz = F.a.z;
#pragma unroll
        for (int d = 0; d < kN; ++d)
        {
            const double t = __builtin_fma(k[d][2], pz, __builtin_fma(k[d][1], py, k[d][0] * px));
            float s, c;
            sincos_turns((float)(t - __builtin_rint(t)), s, c);
#pragma unroll
            for (int q = 0; q < 6; ++q)
            {
                float *a = &acc[d * kV + q * (kV / 6)];
                if (OPP)
                {
                    a[0] = __builtin_fmaf(xr[q], c, a[0]);
                    a[1] = __builtin_fmaf(xi[q], s, a[1]);
                    a[2] = __builtin_fmaf(xi[q], c, a[2]);
                    a[3] = __builtin_fmaf(xr[q], s, a[3]);
                }
                else
                {
                    a[0] = __builtin_fmaf(-xi[q], s, __builtin_fmaf(xr[q], c, a[0]));
                    a[1] = __builtin_fmaf(xr[q], s, __builtin_fmaf(xi[q], c, a[1]));
                }
            }
        }
    }
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int first = wave_sums(acc);
    if (!(lane & 1))
        for (int i = 0; i < 3; ++i)
            wsum[wave][first + i] = acc[i];
    __syncthreads();
    if (threadIdx.x < kSums * kAcc)
    {
        const int v = threadIdx.x / kSums, r = threadIdx.x % kSums;
        const int o = r / kN, d = r % kN;
        const int x = v % 3, ri = (v / 3) & 1, jm = v / 6; // component, re or im, J or M
        float s = 0.f;
        for (int w = 0; w < kFfThreads / 64; ++w)
        {
            const float *a = &wsum[w][d * kV + (jm * 3 + x) * (kV / 6)];
            if (!OPP)
                s += a[ri];
            else if (ri == 0)
                s += o ? a[0] + a[1] : a[0] - a[1];
            else
                s += o ? a[2] - a[3] : a[2] + a[3];
        }
        if (e0 + d < n)
            part[(((long long)fr * kAcc + v) * D.sides() + o) * n + e0 + d] = s;
    }
}

// ---- the faces of a context on their lattice ----

// Places in an array of a lattice's currents: planes one after another, each
// [u][v padded to 8][4 currents].
struct FfLattice : HuyLattice
{
    int np[3];                   // n padded to a tile's 8
    long long off[kHuyPlanes + 1]; // float2 of a plane's currents
    explicit FfLattice(const HuyLattice &h) : HuyLattice(h)
    {
        for (int q = 0; q < 3; ++q)
            np[q] = (n[q] + 7) / 8 * 8;
        off[0] = 0;
        for (int p = 0; p < nplane; ++p)
            off[p + 1] = off[p] + 4LL * n[axis[p] == 0 ? 1 : 0] * np[axis[p] == 2 ? 1 : 2];
    }
    __device__ long long slot(const int co[3], int a) const
    {
        const int u = kTan[a][0], v = kTan[a][1];
        int pl = 0;
        while (pl < nplane - 1 && !(axis[pl] == a && coord[pl] == co[a]))
            ++pl;
        return off[pl] + ((long long)(co[u] - lo[u]) * np[v] + co[v] - lo[v]) * 4;
    }
};

__device__ inline void face_cell(long long p, int nx, long long Pp, int co[3])
{
    const long long k = p / Pp, r = p - k * Pp;
    co[1] = (int)(r / nx);
    co[0] = (int)(r - (long long)co[1] * nx);
    co[2] = (int)k;
}

// Marks the cell coordinates of the faces, used[axis], and of their planes,
// norm[axis] (bytes of the three axes one after another; every writer stores 1).
__global__ void k_huy_used(int nf, const long long *pcell, const int *axis, int nx, int ny, long long Pp,
                           uint8_t *used, uint8_t *norm)
{
    const int f = blockIdx.x * blockDim.x + threadIdx.x;
    if (f >= nf)
        return;
    int co[3];
    face_cell(pcell[f], nx, Pp, co);
    co[1] += nx;
    co[2] += nx + ny;
    for (int q = 0; q < 3; ++q)
        used[co[q]] = 1;
    norm[co[axis[f]]] = 1;
}

// Faces per lattice place: *twice = 1 if a place has two.
__global__ void k_huy_twice(int nf, const long long *pcell, const int *axis, int nx, long long Pp, FfLattice L,
                            int *seen, int *twice)
{
    const int f = blockIdx.x * blockDim.x + threadIdx.x;
    if (f >= nf)
        return;
    int co[3];
    face_cell(pcell[f], nx, Pp, co);
    if (atomicAdd(&seen[L.slot(co, axis[f]) / 4], 1) > 0)
        *twice = 1;
}

// Clears n float4 (13 us as hipMemsetAsync for 13 MB).
__global__ void k_ff_clear(float4 *p, long long n)
{
    for (long long i = blockIdx.x * 256LL + threadIdx.x; i < n; i += gridDim.x * 256LL)
        p[i] = make_float4(0.f, 0.f, 0.f, 0.f);
}

// Currents on the lattice, J_t1, J_t2, M_t1, M_t2 of a place (make_face's; a
// place without a face holds zeros). *odd = 1 if one is not a finite number.
__global__ void k_ff_currents(int nf, const long long *pcell, const int *axis, const float *dft, int nx, int ny,
                              int nz, long long Pp, FfLattice L, float2 *cur, int *odd)
{
    const int f = blockIdx.x * blockDim.x + threadIdx.x;
    if (f >= nf)
        return;
    int co[3];
    face_cell(pcell[f], nx, Pp, co);
    const int a = axis[f], nn = a == 0 ? nx : a == 1 ? ny : nz;
    const float s = ((2 * co[a] + 1 < nn) ? -1.0f : 1.0f) * (a == 1 ? -1.0f : 1.0f);
    const float4 *q = reinterpret_cast<const float4 *>(dft + 8 * (long long)f);
    const float4 e = q[0], h = q[1]; // E1, E2; eta0 H1, eta0 H2
    float4 *o = reinterpret_cast<float4 *>(cur + L.slot(co, a));
    o[0] = make_float4(-s * h.z, -s * h.w, s * h.x, s * h.y);
    o[1] = make_float4(s * e.z, s * e.w, -s * e.x, -s * e.y);
    // 0 times a finite number is 0
    const float z = 0.f * e.x + 0.f * e.y + 0.f * e.z + 0.f * e.w + 0.f * h.x + 0.f * h.y + 0.f * h.z + 0.f * h.w;
    if (z != 0.f)
        *odd = 1;
}

// Phase factors of the axes, rows x, then y, then z: E[r][direction] =
// e^{j 2 pi t}, t the wave vector times the place of coordinate lo + r from the
// middle of the lattice; zero past the last coordinate and direction. (Phases
// from the lattice's middle: a factor common to all faces does not change U.)
__global__ void k_ff_phase(FfLattice L, double dl, FfDirs D, int d0, int pitch, float2 *E)
{
    const int d = blockIdx.x * blockDim.x + threadIdx.x;
    if (d >= pitch)
        return;
    int q = 0, r = blockIdx.y;
    while (q < 2 && r >= L.np[q])
        r -= L.np[q++];
    float2 e = make_float2(0.f, 0.f);
    if (d0 + d < D.n() && r < L.n[q])
    {
        const double t = D.wave(d0 + d, q) * ((r - 0.5 * (L.n[q] - 1)) * dl);
        double s, c;
        sincospi(2.0 * (t - rint(t)), &s, &c);
        e = make_float2((float)c, (float)s);
    }
    E[(long long)blockIdx.y * pitch + d] = e;
}

typedef float f16v __attribute__((ext_vector_type(16)));

// One workgroup: 32 entries e (and their opposites, OPP) and four column
// tiles of a plane, one to a wave; a tile is 8 v by the 4 currents.
// u and its mirror image have conjugate factors (c, -s) and (c, s), so they go
// in together: c (J_lo + J_hi) and j s (J_lo - J_hi), half the products; and
// those two apart give the opposite direction too. A wave's tile is the product
// (32 entries) x (u) with (u) x (32 columns) as four v_mfma_f32_32x32x2_f32 per
// two pairs u. Lane l holds A's row and B's column l % 32 of k = l / 32, and of
// D column l % 32 in rows 8 (i / 4) + 4 (l / 32) + i % 4, i = 0..15.
// Bound by the matrix cores and the loads behind them: 369024 faces x 37 x 73
// directions 1932 us in the sums over faces, 180 with the mirror images
// together, 102 with opposite directions too (50 at the matrix cores' FP32 peak,
// 70 at the rate they reach here without any loads). Three waves a SIMD
// and tiles of 32 entries: 179 against 203 with 64 entries and two waves, 194
// with batches of two row pairs for four.
template <bool OPP>
__global__ void __launch_bounds__(kFfThreads, 3)
    k_ff_lattice(FfLattice L, const float2 *cur, const float2 *E, int pitch, int ndt, int share, float *part)
{
    constexpr int kAhead = 4, kSide = OPP ? 2 : 1;
    __shared__ float red[kFfThreads / 64][kTile][8 * kSide];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int col = lane & 31, half = lane >> 5;
    // workgroups of one XCD (every eighth) share planes, whose currents its L2 keeps
    const int per = gridDim.x / 8, id = (blockIdx.x % 8) * per + blockIdx.x / 8;
    if (id >= ndt * L.nplane * share)
        return;
    const int fr = id / ndt, d0 = (id - fr * ndt) * kTile;
    const int pl = fr / share, t = (fr - pl * share) * (kFfThreads / 64) + wave;
    const int a = L.axis[pl], u = kTan[a][0], v = kTan[a][1];
    const float2 *Ex = E, *Ey = Ex + (long long)L.np[0] * pitch, *Ez = Ey + (long long)L.np[1] * pitch;
    const float2 *Eu = a == 0 ? Ey : Ex, *Ev = a == 2 ? Ey : Ez, *En = a == 0 ? Ex : a == 1 ? Ey : Ez;
    const int nu = L.n[u], npair = (nu + 1) / 2;
    const long long ustride = (long long)L.np[v] * 4;
    if (t < L.np[v] / 8)
    {
        // c Sr, c Si, -s Di, s Dr of S = J_lo + J_hi, D = J_lo - J_hi (added up as
        // they come without opposites)
        f16v m[2 * kSide] = {};
        auto mul = [&](float2 w, float2 x, float2 y) {
            m[0] = __builtin_amdgcn_mfma_f32_32x32x2f32(w.x, x.x + y.x, m[0], 0, 0, 0);
            m[1] = __builtin_amdgcn_mfma_f32_32x32x2f32(w.x, x.y + y.y, m[1], 0, 0, 0);
            m[2 * kSide - 2] = __builtin_amdgcn_mfma_f32_32x32x2f32(w.y, y.y - x.y, m[2 * kSide - 2], 0, 0, 0);
            m[2 * kSide - 1] = __builtin_amdgcn_mfma_f32_32x32x2f32(w.y, x.x - y.x, m[2 * kSide - 1], 0, 0, 0);
        };
        // full batches of kAhead row pairs, the next batch's rows loaded before
        // the present one's products; then pair by pair to the middle
        const float2 *pa = Eu + d0, *plo = cur + L.off[pl] + t * 32, *phi = plo + (nu - 2) * ustride;
        const unsigned oa = half * pitch + col, ol = half * (unsigned)ustride + col,
                       oh = (1 - half) * (unsigned)ustride + col;
        float2 A[kAhead], lo[kAhead], hi[kAhead], An[kAhead], lon[kAhead], hin[kAhead];
        auto load = [&]() {
#pragma unroll
            for (int e = 0; e < kAhead; ++e)
            {
                An[e] = pa[oa];
                lon[e] = plo[ol];
                hin[e] = phi[oh];
                pa += 2 * pitch;
                plo += 2 * ustride;
                phi -= 2 * ustride;
            }
        };
        const int full = nu / 2 / (2 * kAhead);
        if (full > 0)
        {
            load();
            for (int q = 1; q < full; ++q)
            {
#pragma unroll
                for (int e = 0; e < kAhead; ++e)
                {
                    A[e] = An[e];
                    lo[e] = lon[e];
                    hi[e] = hin[e];
                }
                load();
#pragma unroll
                for (int e = 0; e < kAhead; ++e)
                    mul(A[e], lo[e], hi[e]);
            }
#pragma unroll
            for (int e = 0; e < kAhead; ++e)
                mul(An[e], lon[e], hin[e]);
        }
        const float2 *ta = Eu + d0 + col, *tb = cur + L.off[pl] + t * 32 + col;
        for (int q = full * 2 * kAhead; q < npair; q += 2)
        {
            // the middle of an odd number is its own image, and an odd number of
            // pairs leaves the upper half without one
            const int i = min(q + half, npair - 1), k = nu - 1 - i;
            float2 w = ta[(long long)i * pitch], y = tb[k * ustride];
            if (k == i)
                y = make_float2(0.f, 0.f);
            if (q + half >= npair)
                w = make_float2(0.f, 0.f);
            mul(w, tb[i * ustride], y);
        }
        // times the factors of v, over the tile's 8 v, times the plane's factor
        const float2 *pv = Ev + (long long)(t * 8 + (col >> 2)) * pitch + d0 + 4 * half;
        const float2 *pn = En + (long long)(L.coord[pl] - L.lo[a]) * pitch + d0 + 4 * half;
#pragma unroll
        for (int i = 0; i < 16; ++i)
        {
            const int row = 8 * (i >> 2) + (i & 3);
            const float2 f = pv[row], g = pn[row];
#pragma unroll
            for (int o = 0; o < kSide; ++o)
            {
                // the opposite direction has -s for s, in all three factors
                const float sg = o ? -1.f : 1.f;
                const float re = OPP ? __builtin_fmaf(sg, m[2 * kSide - 2][i], m[0][i]) : m[0][i];
                const float im = OPP ? __builtin_fmaf(sg, m[2 * kSide - 1][i], m[1][i]) : m[1][i];
                float x = __builtin_fmaf(-im, sg * f.y, re * f.x), y = __builtin_fmaf(re, sg * f.y, im * f.x);
#pragma unroll
                for (int w = 4; w < 32; w <<= 1)
                {
                    x += __shfl_xor(x, w, 64);
                    y += __shfl_xor(y, w, 64);
                }
                if (col < 4)
                {
                    red[wave][row + 4 * half][8 * o + col] = __builtin_fmaf(-y, sg * g.y, x * g.x);
                    red[wave][row + 4 * half][8 * o + 4 + col] = __builtin_fmaf(x, sg * g.y, y * g.x);
                }
            }
        }
    }
    else
        for (int e = lane; e < kTile * 8 * kSide; e += 64)
            red[wave][e / (8 * kSide)][e % (8 * kSide)] = 0.f;
    __syncthreads();
    // S_J and S_M; their normal components are zero
    for (int e = threadIdx.x; e < kTile * kAcc * kSide; e += kFfThreads)
    {
        const int d = e % kTile, o = e / kTile % kSide, q = e / kTile / kSide;
        const int x = q % 3, ri = (q / 3) & 1, jm = q / 6; // component, re or im, J or M
        float s = 0.f;
        if (x != a)
            for (int w = 0; w < kFfThreads / 64; ++w)
                s += red[w][d][8 * o + 4 * ri + 2 * jm + (x == v ? 1 : 0)];
        part[(((long long)fr * kAcc + q) * kSide + o) * pitch + d0 + d] = s;
    }
}

// U of entries e = d0 + [0, pitch), side blockIdx.y, from the partial sums of
// nfr ranges: 32 entries per workgroup, eight threads to each, which take
// ranges in turn and add up in a fixed order.
__global__ void __launch_bounds__(kFfThreads)
    k_ff_finish(const float *part, int nfr, FfDirs D, int d0, int pitch, float *U)
{
    constexpr int kSlice = kFfThreads / kOut;
    __shared__ double sum[kSlice][kAcc][kOut];
    const int l = threadIdx.x % kOut, w = threadIdx.x / kOut, o = blockIdx.y, no = gridDim.y;
    const int i = blockIdx.x * kOut + l, e = d0 + i;
    const bool on = i < pitch && e < D.n();
    double S[kAcc];
#pragma unroll
    for (int q = 0; q < kAcc; ++q)
        S[q] = 0.0;
    if (on)
        for (int fr = w; fr < nfr; fr += kSlice)
#pragma unroll
            for (int q = 0; q < kAcc; ++q)
                S[q] += part[(((long long)fr * kAcc + q) * no + o) * pitch + i];
#pragma unroll
    for (int q = 0; q < kAcc; ++q)
        sum[w][q][l] = S[q];
    __syncthreads();
    if (w > 0 || !on)
        return;
#pragma unroll
    for (int q = 0; q < kAcc; ++q)
        for (int z = 1; z < kSlice; ++z)
            S[q] += sum[z][q][l];
    const int2 at = D.at(e, o);
    const double2 th = D.ang[at.x], ph = D.ang[D.nT + at.y];
    const double t[3] = {th.x * ph.x, th.x * ph.y, -th.y}, p[2] = {-ph.y, ph.x};
    // radiation vectors projected (J' -> N, M -> L), TlmSolver.cpp:872-889
    const double NtR = S[0] * t[0] + S[1] * t[1] + S[2] * t[2];
    const double NtI = S[3] * t[0] + S[4] * t[1] + S[5] * t[2];
    const double NpR = S[0] * p[0] + S[1] * p[1];
    const double NpI = S[3] * p[0] + S[4] * p[1];
    const double LtR = S[6] * t[0] + S[7] * t[1] + S[8] * t[2];
    const double LtI = S[9] * t[0] + S[10] * t[1] + S[11] * t[2];
    const double LpR = S[6] * p[0] + S[7] * p[1];
    const double LpI = S[9] * p[0] + S[10] * p[1];
    const double aR = LpR + NtR, aI = LpI + NtI;
    const double bR = LtR - NpR, bI = LtI - NpI;
    const float v = (float)(aR * aR + aI * aI + bR * bR + bI * bI);
    float *row = U + at.x * D.nP;
    row[at.y] = v;
    if (D.h && at.y == 0)
        row[D.nP - 1] = v; // phi = 2 pi
}

// Buffers carved in order from a device workspace (256-byte aligned pieces).
struct Carve
{
    unsigned char *base = nullptr;
    size_t off = 0;
    static size_t piece(size_t bytes)
    {
        return (std::max<size_t>(bytes, 1) + 255) / 256 * 256;
    }
    template <class T> T *get(size_t n)
    {
        T *x = reinterpret_cast<T *>(base + off);
        off += piece(n * sizeof(T));
        return x;
    }
};

// Workspace of the allocation-free variant.
constexpr size_t kScratchBytes = (size_t)128 << 20;

// A context keeps its workspace for the next call up to this size (an
// allocation and its release take longer than the other host work of a call).
constexpr size_t kKeep = (size_t)64 << 20;

// One device allocation for a call.
struct DevBuf
{
    unsigned char *p = nullptr;
    ~DevBuf()
    {
        if (p)
            (void)hipFree(p);
    }
};

// Pinned host memory for a call: faces up to kStage bytes go to the device
// through it in one copy (50021 of them: 489 us a call, 533 in copies from
// pageable memory; larger pinned blocks take long to make).
constexpr size_t kStage = (size_t)8 << 20;
struct HostBuf
{
    unsigned char *p = nullptr;
    ~HostBuf()
    {
        if (p)
            (void)hipHostFree(p);
    }
};

// Ranges of nf faces for ngrp groups of k_ff_sums: enough that the grid fills
// the chip, each range at least a block of faces.
int face_ranges(int nf, int ngrp)
{
    return std::max(1, std::min((nf + kFfThreads - 1) / kFfThreads, (2048 + ngrp - 1) / ngrp));
}

// Output directions and what follows the sums.
struct Output
{
    int nT, nP;
    float f0;
    float *U;
    tlm_far_field_summary *out;
    std::vector<double2> ang;
    std::vector<float> u;
    Output(int nT_, int nP_, float f, float *U_, tlm_far_field_summary *o)
        : nT(nT_), nP(nP_), f0(f), U(U_), out(o), ang((size_t)nT_ + nP_), u((size_t)nT_ * nP_)
    {
        // (TlmSolver.cpp:852-861)
        for (int i = 0; i < nT; ++i)
            ang[i] = make_double2(std::cos(M_PI * i / (nT - 1)), std::sin(M_PI * i / (nT - 1)));
        for (int i = 0; i < nP; ++i)
            ang[nT + i] = make_double2(std::cos(2.0 * M_PI * i / (nP - 1)), std::sin(2.0 * M_PI * i / (nP - 1)));
    }
    int ndir() const
    {
        return nT * nP;
    }
    // Device bytes and pieces every transform needs: the angles, U and a flag.
    size_t bytes() const
    {
        return Carve::piece((ang.size() + 1) * sizeof(double2)) + Carve::piece(u.size() * sizeof(float));
    }
    FfDirs dirs(const double2 *d_ang) const
    {
        return FfDirs{d_ang, nT, nP, nP % 2 ? (nP - 1) / 2 : 0, (double)f0 / kC0};
    }
    // directivity and peak (TlmSolver.cpp:893-913)
    void finish() const
    {
        const float PI = (float)M_PI;
        float uMax = 0.0f;
        int iMax = 0;
        double prad = 0.0;
        const float dTh = PI / (nT - 1), dPh = 2.0f * PI / (nP - 1);
        for (int ti = 0; ti < nT; ++ti)
        {
            const float th = PI * ti / (nT - 1);
            const float wTh = (ti == 0 || ti == nT - 1) ? 0.5f : 1.0f;
            const float sth = std::sin(th);
            for (int pi = 0; pi < nP; ++pi)
            {
                const float wPh = (pi == 0 || pi == nP - 1) ? 0.5f : 1.0f;
                const float v = u[(size_t)ti * nP + pi];
                if (v > uMax)
                {
                    uMax = v;
                    iMax = ti * nP + pi;
                }
                prad += (double)v * sth * wTh * wPh * dTh * dPh;
            }
        }
        if (U)
            std::copy(u.begin(), u.end(), U);
        if (out)
        {
            out->u_max = uMax;
            out->directivity = prad > 0 ? (float)(4.0 * M_PI * uMax / prad) : 0.0f;
            out->peak_theta_deg = 180.0f * (iMax / nP) / (nT - 1);
            out->peak_phi_deg = 360.0f * (iMax % nP) / (nP - 1);
        }
    }
};

#define FFCHK(call)                                                                                \
    do                                                                                             \
    {                                                                                              \
        hipError_t e_ = (call);                                                                    \
        if (e_ != hipSuccess)                                                                      \
            return hip_fail(c, e_, #call);                                                         \
    } while (0)

// ---- any faces ----

struct SumsShape
{
    int ngrp, nfr, per;
    size_t part; // partial sums
    SumsShape(int nf, const FfDirs &D)
    {
        const int e = kSums / D.sides();
        ngrp = (D.n() + e - 1) / e;
        nfr = face_ranges(nf, ngrp);
        per = (nf + nfr - 1) / nfr;
        part = (size_t)nfr * kAcc * D.sides() * D.n();
    }
};

size_t sums_bytes(const Output &o, int nf)
{
    return o.bytes() + Carve::piece((size_t)nf * sizeof(FfFace)) +
           Carve::piece(SumsShape(nf, o.dirs(nullptr)).part * sizeof(float));
}

// Sums and U of nf faces, whose records make(faces) queues on stream st; w is
// a workspace of sums_bytes.
template <class Make>
int sums_transform(tlm_ctx *c, hipStream_t st, unsigned char *w, int nf, Output &o, Make make)
{
    Carve b{w};
    double2 *d_ang = b.get<double2>(o.ang.size() + 1);
    float *d_U = b.get<float>(o.u.size());
    FfFace *faces = b.get<FfFace>((size_t)nf);
    const FfDirs D = o.dirs(d_ang);
    const SumsShape S(nf, D);
    float *part = b.get<float>(S.part);
    FFCHK(hipMemcpyAsync(d_ang, o.ang.data(), o.ang.size() * sizeof(double2), hipMemcpyHostToDevice, st));
    make(faces);
    FFCHK(hipGetLastError());
    (D.h ? k_ff_sums<true> : k_ff_sums<false>)<<<dim3((unsigned)S.ngrp, (unsigned)S.nfr), kFfThreads, 0, st>>>(
        faces, nf, S.per, D, part);
    FFCHK(hipGetLastError());
    k_ff_finish<<<dim3((unsigned)((D.n() + kOut - 1) / kOut), (unsigned)D.sides()), kFfThreads, 0, st>>>(
        part, S.nfr, D, 0, D.n(), d_U);
    FFCHK(hipGetLastError());
    FFCHK(hipMemcpyAsync(o.u.data(), d_U, o.u.size() * sizeof(float), hipMemcpyDeviceToHost, st));
    FFCHK(hipStreamSynchronize(st));
    return TLM_OK;
}

// ---- a context's box ----

// Shape of the transform on a lattice: directions go in batches whose phase
// tables and partial sums stay within kTables.
constexpr size_t kTables = (size_t)24 << 20;
struct LatticeShape
{
    FfLattice L;
    int share = 1, nfr = 0, pitch = 0; // workgroups a plane and a tile of directions
    size_t rows = 0, part = 0;
    LatticeShape(const HuyLattice &h, const FfDirs &D) : L(h)
    {
        int ntile = 1;
        for (int q = 0; q < 3; ++q)
            rows += L.np[q];
        for (int p = 0; p < L.nplane; ++p)
            ntile = std::max(ntile, L.np[L.axis[p] == 2 ? 1 : 2] / 8);
        const int ndt = (D.n() + kTile - 1) / kTile, waves = kFfThreads / 64;
        share = (ntile + waves - 1) / waves;
        nfr = L.nplane * share;
        const size_t sums = (size_t)nfr * kAcc * D.sides(), per = rows * sizeof(float2) + sums * sizeof(float);
        const int most = (int)std::max<size_t>(1, std::min<size_t>(kTables / per / kTile, (size_t)ndt));
        const int batches = (ndt + most - 1) / most;
        pitch = (ndt + batches - 1) / batches * kTile;
        part = sums * pitch;
    }
    size_t cur() const
    {
        return (size_t)L.off[L.nplane];
    }
    size_t bytes(const Output &o) const
    {
        return o.bytes() + Carve::piece(cur() * sizeof(float2)) + Carve::piece(rows * pitch * sizeof(float2)) +
               Carve::piece(part * sizeof(float));
    }
};

// The same over the lattice of c's faces. *odd: a current is not a finite
// number, which a product with the zeros of the padding would spread (U is then
// to be taken from k_ff_sums).
int lattice_transform(tlm_ctx *c, unsigned char *w, const LatticeShape &S, Output &o, bool *odd)
{
    hipStream_t st = c->stream;
    Carve b{w};
    double2 *d_ang = b.get<double2>(o.ang.size() + 1);
    int *d_odd = reinterpret_cast<int *>(d_ang + o.ang.size());
    float *d_U = b.get<float>(o.u.size());
    float2 *cur = b.get<float2>(S.cur()), *E = b.get<float2>(S.rows * S.pitch);
    float *part = b.get<float>(S.part);
    std::vector<double2> ang(o.ang);
    ang.push_back(make_double2(0.0, 0.0)); // clears the flag
    FFCHK(hipMemcpyAsync(d_ang, ang.data(), ang.size() * sizeof(double2), hipMemcpyHostToDevice, st));
    k_ff_clear<<<(unsigned)std::min<size_t>(S.cur() / 512 + 1, 4096), 256, 0, st>>>(
        reinterpret_cast<float4 *>(cur), (long long)(S.cur() / 2)); // cur() is a multiple of 32
    FFCHK(hipGetLastError());
    k_ff_currents<<<(c->nh + 255) / 256, 256, 0, st>>>(c->nh, c->hcell, c->haxis, c->huy8, c->nx, c->ny, c->nz,
                                                       c->Pp, S.L, cur, d_odd);
    FFCHK(hipGetLastError());
    const FfDirs D = o.dirs(d_ang);
    for (int d0 = 0; d0 < D.n(); d0 += S.pitch)
    {
        const int ndt = (std::min(S.pitch, D.n() - d0) + kTile - 1) / kTile;
        k_ff_phase<<<dim3((unsigned)((S.pitch + 255) / 256), (unsigned)S.rows), 256, 0, st>>>(
            S.L, (double)c->dl, D, d0, S.pitch, E);
        FFCHK(hipGetLastError());
        (D.h ? k_ff_lattice<true> : k_ff_lattice<false>)<<<(unsigned)(ndt * S.nfr + 7) / 8 * 8, kFfThreads, 0, st>>>(
            S.L, cur, E, S.pitch, ndt, S.share, part);
        FFCHK(hipGetLastError());
        k_ff_finish<<<dim3((unsigned)(ndt * kTile / kOut), (unsigned)D.sides()), kFfThreads, 0, st>>>(
            part, S.nfr, D, d0, S.pitch, d_U);
        FFCHK(hipGetLastError());
    }
    int flag = 0;
    FFCHK(hipMemcpyAsync(&flag, d_odd, sizeof(int), hipMemcpyDeviceToHost, st));
    FFCHK(hipMemcpyAsync(o.u.data(), d_U, o.u.size() * sizeof(float), hipMemcpyDeviceToHost, st));
    FFCHK(hipStreamSynchronize(st));
    *odd = flag != 0;
    return TLM_OK;
}

// From this many faces times sums the lattice is faster than k_ff_sums, whose
// time is theirs, where the lattice's four more passes take some 40 us at any
// size: 37 x 73 directions 31104 faces 109 us a call against 103, 62424 121
// against 155; 91 x 181 6144 141 against 123, 13824 166 against 191; 37 x 72
// 13824 102 against 92, 31104 120 against 140.
constexpr double kLatticeTerms = 5e7;

// Finds whether the context's faces are the places of a few planes of a box
// (each once, and most of them there) and records its extent: at the first
// transform of a list that may use it, in the transform's workspace w of
// scan_bytes (at tlm_set_huygens it took 40 us, 64^3, of callers who take no far
// field).
size_t scan_marks(const tlm_ctx *c)
{
    return Carve::piece(2 * (size_t)(c->nx + (long long)c->ny + c->nz));
}
size_t scan_bytes(const tlm_ctx *c)
{
    return scan_marks(c) + Carve::piece(((size_t)c->nh * 3 / 2 + 1) * sizeof(int)); // huy_lattice_fits
}
int huy_lattice_scan(tlm_ctx *c, unsigned char *w)
{
    c->hlat = HuyLattice{};
    c->hlat_known = true;
    const int n = c->nh;
    const size_t len = (size_t)c->nx + c->ny + c->nz;
    hipStream_t st = c->stream;
    HuyLattice h;
    FFCHK(hipMemsetAsync(w, 0, 2 * len, st));
    k_huy_used<<<(n + 255) / 256, 256, 0, st>>>(n, c->hcell, c->haxis, c->nx, c->ny, c->Pp, w, w + len);
    FFCHK(hipGetLastError());
    std::vector<uint8_t> m(2 * len);
    FFCHK(hipMemcpyAsync(m.data(), w, m.size(), hipMemcpyDeviceToHost, st));
    FFCHK(hipStreamSynchronize(st));
    const int dims[3] = {c->nx, c->ny, c->nz};
    size_t at = 0;
    for (int q = 0; q < 3; at += dims[q], ++q)
    {
        int lo = 0, hi = dims[q] - 1;
        while (lo < hi && !m[at + lo])
            ++lo;
        while (hi > lo && !m[at + hi])
            --hi;
        h.lo[q] = lo;
        h.n[q] = hi - lo + 1;
        for (int i = lo; i <= hi; ++i)
            if (m[len + at + i])
            {
                if (h.nplane == kHuyPlanes)
                    return TLM_OK;
                h.axis[h.nplane] = q;
                h.coord[h.nplane++] = i;
            }
    }
    if (!huy_lattice_fits(h, n))
        return TLM_OK;
    const FfLattice L(h);
    const size_t places = (size_t)L.off[L.nplane] / 4;
    int *cnt = reinterpret_cast<int *>(w + scan_marks(c)), twice = 0;
    FFCHK(hipMemsetAsync(cnt, 0, (places + 1) * sizeof(int), st));
    k_huy_twice<<<(n + 255) / 256, 256, 0, st>>>(n, c->hcell, c->haxis, c->nx, c->Pp, L, cnt, cnt + places);
    FFCHK(hipGetLastError());
    FFCHK(hipMemcpyAsync(&twice, cnt + places, sizeof(int), hipMemcpyDeviceToHost, st));
    FFCHK(hipStreamSynchronize(st));
    h.ok = !twice;
    c->hlat = h;
    return TLM_OK;
}

// Both entry points of a context: ws(bytes, &p) gives the workspace.
template <class Ws> int ctx_transform(tlm_ctx *c, const float origin[3], Output &o, Ws ws)
{
    unsigned char *w = nullptr;
    int rc;
    const bool many = c->nh >= kHuyLatticeMin && (double)c->nh * o.dirs(nullptr).n() >= kLatticeTerms &&
                      std::isfinite(origin[0]) && std::isfinite(origin[1]) && std::isfinite(origin[2]);
    if (many && !c->hlat_known && scan_bytes(c) <= kScratchBytes)
    {
        if ((rc = ws(scan_bytes(c), &w)) || (rc = huy_lattice_scan(c, w)))
            return rc;
    }
    if (many && c->hlat.ok)
    {
        const LatticeShape S(c->hlat, o.dirs(nullptr));
        bool odd = false;
        if ((rc = ws(S.bytes(o), &w)) || (rc = lattice_transform(c, w, S, o, &odd)))
            return rc;
        if (!odd)
        {
            o.finish();
            return TLM_OK;
        }
    }
    if ((rc = ws(sums_bytes(o, c->nh), &w)))
        return rc;
    rc = sums_transform(c, c->stream, w, c->nh, o, [&](FfFace *faces) {
        k_ff_faces_ctx<<<(c->nh + 255) / 256, 256, 0, c->stream>>>(c->nh, c->hcell, c->haxis, c->huy8, c->nx, c->ny,
                                                                   c->nz, c->Pp, origin[0], origin[1], origin[2],
                                                                   c->dl, faces);
    });
    if (!rc)
        o.finish();
    return rc;
}

// ---- allocation-free variant ----
// Its workspace: a file-scope device array of kScratchBytes, one instance per
// GPU the library runs on (held until the process ends). Host code reaches
// it only through the address hipGetSymbolAddress gives on each device.
constexpr int kMaxDevices = 64;

// Its size beyond kScratchBytes: face_ranges may split the faces finer for the
// fewer groups of k_ff_sums<true>, at most 32768 sums of 48 bytes more.
constexpr size_t kScratchSlack = (size_t)2 << 20;

// What it takes: nf faces and ndir directions whose k_ff_sums with its inputs
// as float tables (64 bytes a face, 52 a direction and 48 a direction and
// range) fits. k_ff_sums needs less, and so does the lattice: at most 48 bytes a
// face (huy_lattice_fits), 4 a direction, and kTables.
size_t far_field_workspace(int nf, int ndir)
{
    const size_t nfr = (size_t)face_ranges(nf, (ndir + 7) / 8);
    return Carve::piece((size_t)nf * sizeof(FfFace)) + Carve::piece(9 * (size_t)ndir * sizeof(float)) +
           Carve::piece(3 * (size_t)ndir * sizeof(float)) +
           Carve::piece((size_t)ndir * nfr * kAcc * sizeof(float)) + Carve::piece((size_t)ndir * sizeof(float));
}

__device__ __align__(256) unsigned char scratch[kScratchBytes + kScratchSlack];

std::mutex g_scratch_mu;
unsigned char *g_scratch[kMaxDevices] = {};

// Device address of the workspace on device dev, which must be current;
// looked up once per device.
int scratch_on(tlm_ctx *c, int dev, unsigned char **out)
{
    if (dev < 0 || dev >= kMaxDevices)
        return fail(c, TLM_ERR_UNSUPPORTED, "allocation-free far field: device ordinal above 63");
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch[dev])
    {
        void *p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p)
            return hip_fail(c, e != hipSuccess ? e : hipErrorInvalidSymbol, "hipGetSymbolAddress(scratch)");
        g_scratch[dev] = static_cast<unsigned char *>(p);
    }
    *out = g_scratch[dev];
    return TLM_OK;
}

} // namespace

extern "C" {

int tlm_far_field(int device, int nf, const float *pos, const int32_t *axis,
                  const int32_t *out_sign, const float *dft8, int samples, float f0, int n_theta,
                  int n_phi, float *U, tlm_far_field_summary *out)
{
    tlm_ctx *c = nullptr; // errors go to tlm_last_error(NULL)
    if (nf < 0 || n_theta < 2 || n_phi < 2 || (nf > 0 && (!pos || !axis || !out_sign || !dft8)))
        return fail(nullptr, TLM_ERR_ARG, "tlm_far_field: bad arguments");
    if (nf == 0 || samples == 0)
        return fail(nullptr, TLM_ERR_STATE, "tlm_far_field: no Huygens data");
    bool bad = false;
    for (int f = 0; f < nf; ++f)
        bad |= (unsigned)axis[f] > 2u || (out_sign[f] != 1 && out_sign[f] != -1);
    if (bad)
        return fail(nullptr, TLM_ERR_ARG, "tlm_far_field: face axis or sign out of range");
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0)
        return fail(nullptr, TLM_ERR_NO_DEVICE, "no HIP device");
    if (device < 0 || device >= ndev)
        return fail(nullptr, TLM_ERR_ARG, "tlm_far_field: device out of range");
    FFCHK(hipSetDevice(device));
    hipStream_t st;
    FFCHK(hipStreamCreateWithFlags(&st, hipStreamNonBlocking));
    Output o(n_theta, n_phi, f0, U, out);
    int rc = TLM_OK;
    {
        // the faces as given, then the transform's workspace
        const size_t bp = Carve::piece(3 * (size_t)nf * sizeof(float)), bd = Carve::piece(8 * (size_t)nf * sizeof(float)),
                     in = bp + bd + Carve::piece((size_t)nf);
        DevBuf b;
        HostBuf h;
        std::vector<uint8_t> side((size_t)nf);
        for (int f = 0; f < nf; ++f)
            side[f] = (uint8_t)(axis[f] | (out_sign[f] < 0 ? 4 : 0));
        hipError_t e = hipMalloc((void **)&b.p, in + sums_bytes(o, nf));
        if (e == hipSuccess && in <= kStage && hipHostMalloc((void **)&h.p, in, hipHostMallocDefault) != hipSuccess)
        {
            (void)hipGetLastError();
            h.p = nullptr;
        }
        if (e != hipSuccess)
            rc = hip_fail(nullptr, e, "hipMalloc");
        else
        {
            auto put = [&](size_t at, const void *src, size_t n) {
                if (h.p)
                    std::memcpy(h.p + at, src, n);
                else
                    (void)hipMemcpyAsync(b.p + at, src, n, hipMemcpyHostToDevice, st);
            };
            put(0, pos, 3 * (size_t)nf * sizeof(float));
            put(bp, dft8, 8 * (size_t)nf * sizeof(float));
            put(bp + bd, side.data(), (size_t)nf);
            if (h.p)
                (void)hipMemcpyAsync(b.p, h.p, in, hipMemcpyHostToDevice, st);
            rc = sums_transform(nullptr, st, b.p + in, nf, o, [&](FfFace *faces) {
                k_ff_faces_host<<<(nf + 255) / 256, 256, 0, st>>>(nf, reinterpret_cast<const float *>(b.p),
                                                                  b.p + bp + bd,
                                                                  reinterpret_cast<const float *>(b.p + bp), faces);
            });
            (void)hipStreamSynchronize(st); // before side and h go, also after a failure
        }
    }
    (void)hipStreamDestroy(st);
    if (!rc)
        o.finish();
    return rc;
}

int tlm_far_field_ctx(tlm_ctx *c, const float origin[3], int samples, float f0, int n_theta,
                      int n_phi, float *U, tlm_far_field_summary *out)
{
    if (!c || !origin || n_theta < 2 || n_phi < 2)
        return fail(c, TLM_ERR_ARG, "tlm_far_field_ctx: bad arguments");
    if (c->nh == 0 || samples == 0)
        return fail(c, TLM_ERR_STATE, "tlm_far_field_ctx: no Huygens data");
    FFCHK(hipSetDevice(c->dev));
    Output o(n_theta, n_phi, f0, U, out);
    const int rc = ctx_transform(c, origin, o, [&](size_t bytes, unsigned char **p) {
        if (bytes > c->ff_bytes)
        {
            dfree(c, c->ff_ws);
            c->ff_bytes = 0;
            const int e = dalloc(c, &c->ff_ws, bytes);
            if (e)
                return e;
            c->ff_bytes = bytes;
        }
        *p = c->ff_ws;
        return (int)TLM_OK;
    });
    if (c->ff_bytes > kKeep)
    {
        dfree(c, c->ff_ws);
        c->ff_bytes = 0;
    }
    return rc;
}

int tlm_far_field_ctx_noalloc(tlm_ctx *c, const float origin[3], int samples, float f0, int n_theta,
                              int n_phi, float *U, tlm_far_field_summary *out)
{
    if (!c || !origin || n_theta < 2 || n_phi < 2)
        return fail(c, TLM_ERR_ARG, "tlm_far_field_ctx_noalloc: bad arguments");
    if (c->nh == 0 || samples == 0)
        return fail(c, TLM_ERR_STATE, "tlm_far_field_ctx_noalloc: no Huygens data");
    const size_t need = far_field_workspace(c->nh, n_theta * n_phi);
    if (need > kScratchBytes)
        return fail(c, TLM_ERR_UNSUPPORTED,
                    "tlm_far_field_ctx_noalloc: " + std::to_string(c->nh) + " faces x " +
                        std::to_string(n_theta * n_phi) + " directions need " + std::to_string(need) +
                        " bytes of workspace, above its fixed " + std::to_string(kScratchBytes) +
                        " (tlm_far_field_ctx allocates what it needs)");
    FFCHK(hipSetDevice(c->dev));
    unsigned char *w = nullptr;
    int rc = scratch_on(c, c->dev, &w);
    if (rc)
        return rc;
    Output o(n_theta, n_phi, f0, U, out);
    return ctx_transform(c, origin, o, [&](size_t bytes, unsigned char **p) {
        *p = w;
        return bytes <= kScratchBytes + kScratchSlack ? (int)TLM_OK
                                      : fail(c, TLM_ERR_UNSUPPORTED, "allocation-free far field: workspace");
    });
}

} // extern "C"
