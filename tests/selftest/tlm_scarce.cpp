//---------------------------------------------------------------------------
// tlm_scarce.cpp - the library without memory or threads to spare.
//
// The program defines hipMalloc, hipHostMalloc, hipMemGetInfo and
// pthread_create itself; the library's calls come here, are counted, and are
// refused where a section says so (no device memory is taken to make it
// scarce). Each section's result has to be, bit for bit, the one that the
// library gives with all it asks for:
//   * a context without room for the second stub buffer of pairs of steps takes
//     single steps, without an error left behind, and pairs again after an
//     upload that finds room;
//   * an upload without memory for the device map, refused or not; an upload that
//     fails half way, which leaves nothing to run;
//   * a state read back without pinned memory or without threads, and a small
//     one, which asks for neither;
//   * face lists read without device memory for their order, and the first few
//     faces of one, which ask for none;
//   * a list of Huygens faces set without work for a far field that may not come.
// Prints PASS/FAIL lines and exits 1 on a failure; SKIP without a device.
//---------------------------------------------------------------------------
#include "GpuTlmHip.h"

#include <algorithm>
#include <cerrno>
#include <cstdio>
#include <cstring>
#include <dlfcn.h>
#include <pthread.h>
#include <random>
#include <string>
#include <vector>

namespace {

constexpr size_t kNone = ~(size_t)0;
size_t g_refuse = kNone;     // device allocations of this many bytes or more ...
size_t g_refuse_size = kNone; // ... or of just this many are refused
bool g_no_pinned = false, g_no_threads = false;
size_t g_free = kNone; // free memory to report, if set
int g_mallocs = 0, g_pinned = 0, g_threads = 0;

template <class F> F next(const char *name)
{
    return reinterpret_cast<F>(dlsym(RTLD_NEXT, name));
}

} // namespace

extern "C" int hipMalloc(void **p, size_t n)
{
    static const auto f = next<int (*)(void **, size_t)>("hipMalloc");
    ++g_mallocs;
    if (n >= g_refuse || n == g_refuse_size)
        return 2; // hipErrorOutOfMemory
    return f(p, n);
}

extern "C" int hipHostMalloc(void **p, size_t n, unsigned flags)
{
    static const auto f = next<int (*)(void **, size_t, unsigned)>("hipHostMalloc");
    ++g_pinned;
    return g_no_pinned ? 2 : f(p, n, flags);
}

extern "C" int hipMemGetInfo(size_t *fr, size_t *total)
{
    static const auto f = next<int (*)(size_t *, size_t *)>("hipMemGetInfo");
    const int e = f(fr, total);
    if (e == 0 && g_free != kNone)
        *fr = g_free;
    return e;
}

extern "C" int pthread_create(pthread_t *t, const pthread_attr_t *a, void *(*fn)(void *), void *arg) noexcept
{
    static const auto f = next<int (*)(pthread_t *, const pthread_attr_t *, void *(*)(void *), void *)>("pthread_create");
    ++g_threads;
    return g_no_threads ? EAGAIN : f(t, a, fn, arg);
}

namespace {

int g_fail = 0;

void check(bool ok, const char *what, long long a = 0, long long b = 0)
{
    std::printf("%s  %-66s (%lld / %lld)\n", ok ? "PASS" : "FAIL", what, a, b);
    std::fflush(stdout);
    if (!ok)
        ++g_fail;
}

void must(int rc, const tlm_ctx *c, const char *what)
{
    if (rc < 0)
        check(false, (std::string(what) + ": " + tlm_last_error(c)).c_str(), rc);
}

// A box of dielectric and scattered PEC cells in 70 x 61 x 37 cells (7.6 MB of
// pulses: read back in four chunks), everything random.
constexpr int kNx = 70, kNy = 61, kNz = 37, kCells = kNx * kNy * kNz, kSteps = 24;
constexpr size_t kStubs = (size_t)(kNx * kNy + 63) / 64 * 64 * kNz * 12; // bytes of a stub buffer
std::vector<uint8_t> g_mat(kCells), g_bad;
std::vector<float> g_V(12 * kCells), g_Vs(3 * kCells);
const float kY[1] = {8.0f}, kG[1] = {0.1f};

struct State
{
    std::vector<float> V = std::vector<float>(12 * kCells), Vs = std::vector<float>(3 * kCells);
    bool operator==(const State &o) const
    {
        return std::memcmp(V.data(), o.V.data(), V.size() * 4) == 0 && std::memcmp(Vs.data(), o.Vs.data(), Vs.size() * 4) == 0;
    }
};

tlm_ctx *make()
{
    tlm_grid_desc d = {};
    d.nx = kNx;
    d.ny = kNy;
    d.nz = kNz;
    d.dl = 0.01f;
    d.rho = 0.37f;
    tlm_ctx *c = nullptr;
    if (tlm_create(&d, &c) != TLM_OK)
        return nullptr;
    std::vector<float> z(2 * kSteps, 0.0f);
    must(tlm_set_schedule(c, z.data(), z.data(), z.data(), 2 * kSteps, 0), c, "tlm_set_schedule");
    return c;
}

int upload(tlm_ctx *c, const std::vector<uint8_t> &mat = g_mat)
{
    return tlm_upload(c, mat.data(), kY, kG, 1, g_V.data(), g_Vs.data());
}

void run(tlm_ctx *c, int step0, int n)
{
    must(tlm_run(c, step0, n), c, "tlm_run");
    must(tlm_sync(c), c, "tlm_sync");
}

State read(tlm_ctx *c)
{
    State s;
    must(tlm_read_state(c, s.V.data(), s.Vs.data()), c, "tlm_read_state");
    return s;
}

long long pairs(const tlm_ctx *c)
{
    int64_t n = 0, p = 0;
    must(tlm_step_launches(c, &n, &p), c, "tlm_step_launches");
    return p;
}

void no_second_stub_buffer(const State &ref)
{
    for (int way = 0; way < 2; ++way)
    {
        tlm_ctx *c = make();
        must(upload(c), c, "tlm_upload");
        const std::string before = tlm_last_error(c);
        if (way == 0)
            g_free = 4 * kStubs - 1; // more than a quarter of what is free
        else
            g_refuse = kStubs;
        run(c, 0, kSteps);
        g_free = g_refuse = kNone;
        check(pairs(c) == 0, "no room for a second stub buffer: single steps", pairs(c));
        check(read(c) == ref, "... the same state");
        check(before == tlm_last_error(c), "... and no error left behind");
        must(upload(c), c, "tlm_upload");
        run(c, 0, kSteps);
        check(pairs(c) == kSteps / 2, "an upload that finds room: pairs again", pairs(c), kSteps / 2);
        check(read(c) == ref, "... the same state");
        tlm_destroy(c);
    }
}

void no_map(const State &ref)
{
    tlm_ctx *c = make();
    must(upload(c), c, "tlm_upload");
    run(c, 0, 7);
    g_refuse_size = kCells;
    must(upload(c), c, "tlm_upload");
    run(c, 0, kSteps);
    g_refuse_size = kNone;
    check(read(c) == ref, "an upload without memory for the map");
    must(upload(c), c, "tlm_upload");
    run(c, 0, 9);
    g_refuse_size = kCells;
    const int rc = upload(c, g_bad);
    g_refuse_size = kNone;
    check(rc == TLM_ERR_ARG, "a refused upload without memory for the map", rc, TLM_ERR_ARG);
    run(c, 9, kSteps - 9);
    check(read(c) == ref, "... leaves the state as it was");
    tlm_destroy(c);
}

// A second upload that finds no room for the stubs, or for the block flags.
void failed_upload(const State &ref)
{
    const size_t flags = (size_t)((kNx * kNy + 63) / 64 * kNz + 3) / 4 * 4;
    for (size_t refused : {kStubs, flags})
    {
        tlm_ctx *c = make();
        must(upload(c), c, "tlm_upload");
        run(c, 0, 10);
        g_refuse_size = refused;
        const int rc = upload(c);
        g_refuse_size = kNone;
        check(rc == TLM_ERR_NOMEM, "an upload without room", rc, TLM_ERR_NOMEM);
        const int ran = tlm_run(c, 10, 2);
        check(ran == TLM_ERR_STATE, "... leaves nothing to run", ran, TLM_ERR_STATE);
        (void)read(c);
        must(upload(c), c, "tlm_upload");
        run(c, 0, kSteps);
        check(read(c) == ref, "... and the next one all of it");
        tlm_destroy(c);
    }
}

void no_pinned_or_threads(const State &ref)
{
    tlm_ctx *c = make();
    must(upload(c), c, "tlm_upload");
    run(c, 0, kSteps);
    const int pinned = g_pinned, threads = g_threads;
    check(read(c) == ref, "a state read back");
    check(g_pinned > pinned && g_threads > threads, "... through pinned memory by threads", g_pinned - pinned,
          g_threads - threads);
    g_no_pinned = true;
    check(read(c) == ref, "... without pinned memory");
    g_no_threads = true;
    check(read(c) == ref, "... without threads either");
    g_no_pinned = false;
    check(read(c) == ref, "... without threads");
    g_no_threads = false;
    tlm_destroy(c);
}

void small_state()
{
    tlm_grid_desc d = {};
    d.nx = d.ny = d.nz = 32;
    d.dl = 0.01f;
    tlm_ctx *c = nullptr;
    must(tlm_create(&d, &c), nullptr, "tlm_create");
    const int n = 32 * 32 * 32;
    const std::vector<uint8_t> mat((size_t)n, 2);
    const int mallocs = g_mallocs;
    must(tlm_upload(c, mat.data(), kY, kG, 1, nullptr, nullptr), c, "tlm_upload");
    check(g_mallocs - mallocs == 3, "a small map: block flags, materials and stubs allocated, no more", g_mallocs - mallocs, 3);
    must(tlm_upload(c, mat.data(), kY, kG, 1, g_V.data(), g_Vs.data()), c, "tlm_upload");
    State s;
    const int pinned = g_pinned, threads = g_threads;
    must(tlm_read_state(c, s.V.data(), s.Vs.data()), c, "tlm_read_state");
    check(std::memcmp(s.V.data(), g_V.data(), 12 * n * sizeof(float)) == 0 &&
              std::memcmp(s.Vs.data(), g_Vs.data(), 3 * n * sizeof(float)) == 0,
          "a state of 2 MB read back");
    check(g_pinned == pinned && g_threads == threads, "... without pinned memory or threads", g_pinned - pinned,
          g_threads - threads);
    tlm_destroy(c);
}

void no_list_memory()
{
    tlm_ctx *c = make();
    std::vector<uint8_t> mat(kCells); // a PEC cell in every second one: 62000 faces and more
    for (int q = 0; q < kCells; ++q)
        mat[q] = (q / kNx + q / (kNx * kNy)) % 2 == 0 && q % 2 == 0;
    must(tlm_mat_write(c, mat.data()), c, "tlm_mat_write");
    must(tlm_upload_mat(c, nullptr, nullptr, 0), c, "tlm_upload_mat");
    const int64_t n = tlm_pec_faces_mat(c);
    std::vector<int64_t> a((size_t)n), b((size_t)n);
    std::vector<int32_t> ax((size_t)n), bx((size_t)n);
    must((int)tlm_read_faces(c, a.data(), ax.data(), n), c, "tlm_read_faces");
    g_refuse = 0;
    must((int)tlm_read_faces(c, b.data(), bx.data(), n), c, "tlm_read_faces");
    g_refuse = kNone;
    check(n > 62000 && a == b && ax == bx, "a list read without device memory", n);
    const int mallocs = g_mallocs;
    for (int64_t few : {(int64_t)1, (int64_t)777, (int64_t)4096})
    {
        std::vector<int64_t> d((size_t)few);
        std::vector<int32_t> dx((size_t)few);
        must((int)tlm_read_faces(c, d.data(), dx.data(), few), c, "tlm_read_faces");
        check(std::equal(d.begin(), d.end(), a.begin()) && std::equal(dx.begin(), dx.end(), ax.begin()),
              "the first faces of a list", few);
    }
    check(g_mallocs == mallocs, "... without an allocation", g_mallocs - mallocs);
    tlm_destroy(c);
}

// Setting a list of faces takes the same allocations whatever its length.
void huygens_list()
{
    tlm_ctx *c = make();
    must(upload(c), c, "tlm_upload");
    int took[2] = {};
    for (int k = 0; k < 2; ++k)
    {
        std::vector<int64_t> cells;
        std::vector<int32_t> axes;
        for (int q = 0; q < (k ? 3 * kNx * kNy / 2 : 100); ++q) // 6405 faces
        {
            cells.push_back(q);
            axes.push_back(2);
        }
        const int mallocs = g_mallocs;
        must(tlm_set_huygens(c, cells.data(), axes.data(), (int)cells.size()), c, "tlm_set_huygens");
        took[k] = g_mallocs - mallocs;
    }
    check(took[0] == took[1], "allocations for a list of 100 and of 6405 Huygens faces", took[0], took[1]);
    tlm_destroy(c);
}

} // namespace

int main()
{
    if (tlm_device_count() == 0)
    {
        std::printf("SKIP  no HIP device\n");
        return 0;
    }
    std::mt19937 r(5);
    for (auto &m : g_mat)
        m = r() % 16 == 0;
    for (int k = 10; k < 30; ++k)
        for (int j = 20; j < 50; ++j)
            for (int i = 8; i < 40; ++i)
                g_mat[(k * kNy + j) * kNx + i] = 2;
    g_bad = g_mat;
    g_bad[kCells / 2] = 9;
    std::uniform_real_distribution<float> u(-1.0f, 1.0f);
    for (auto *v : {&g_V, &g_Vs})
        for (auto &x : *v)
            x = u(r);
    for (int q = 0; q < kCells; ++q)
        if (g_mat[q] == 1)
            std::memset(&g_V[12 * (size_t)q], 0, 12 * sizeof(float));

    tlm_ctx *c = make();
    if (!c)
    {
        std::printf("FAIL  tlm_create: %s\n", tlm_last_error(nullptr));
        return 1;
    }
    must(upload(c), c, "tlm_upload");
    run(c, 0, kSteps);
    check(pairs(c) == kSteps / 2, "with memory: pairs", pairs(c), kSteps / 2);
    const State ref = read(c);
    tlm_destroy(c);
    check(g_mallocs > 0, "the library's allocations come here", g_mallocs);

    no_second_stub_buffer(ref);
    no_map(ref);
    failed_upload(ref);
    no_pinned_or_threads(ref);
    small_state();
    no_list_memory();
    huygens_list();
    std::printf(g_fail ? "SCARCETEST FAILED\n" : "SCARCETEST PASSED\n");
    return g_fail ? 1 : 0;
}
