// Host code of libtetemoko_hip checked from the inside: this file is the library's main source with a
// driver below it, built host only with the sanitizers and run against the host-memory stand-in of the HIP
// runtime (hip_host_stand_in.cpp), so that tables a launch would read are plain host memory.  No kernel
// runs.  Usage: host_library CHECK (see main).
#include "../../tetemoko_amd/csrc/tmk_api.hip"

#include <atomic>
#include <cstdlib>
#include <new>
#include <utility>

// operator new throws once this many more allocations have been made on the thread (-1: never)
static thread_local int g_new_left = -1;
void* operator new(std::size_t n)
{
    if (g_new_left == 0) throw std::bad_alloc();
    if (g_new_left > 0) --g_new_left;
    if (void* p = std::malloc(n ? n : 1)) return p;
    throw std::bad_alloc();
}
void* operator new(std::size_t n, const std::nothrow_t&) noexcept
{
    if (g_new_left == 0) return nullptr;
    if (g_new_left > 0) --g_new_left;
    return std::malloc(n ? n : 1);
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, std::size_t) noexcept { std::free(p); }

// the pinned-memory calls, counted (out of memory until a check turns them on: with a stage, a drop-in
// call's error word comes from a kernel), and the current device of a thread (the stand-in's own is weak here)
static std::atomic<int> g_pinned{0}, g_pins{0}, g_frees{0};
static bool g_pin_on = false;
static thread_local int g_dev = 0;
extern "C" {
hipError_t hipHostMalloc(void** p, size_t n, unsigned)
{
    if (!g_pin_on) return hipErrorOutOfMemory;
    *p = std::calloc(n, 1);
    ++g_pins;
    ++g_pinned;
    return hipSuccess;
}
hipError_t hipHostFree(void* p)
{
    std::free(p);
    ++g_frees;
    --g_pinned;
    return hipSuccess;
}
hipError_t hipSetDevice(int dev) { g_dev = dev; return hipSuccess; }
hipError_t hipGetDevice(int* dev) { *dev = g_dev; return hipSuccess; }
}

static void fail(const char* what, int line)
{
    fprintf(stderr, "host_library.cpp:%d: %s\n", line, what);
    exit(1);
}
#define EXPECT(x)                                   \
    do {                                            \
        if (!(x)) fail(#x, __LINE__);               \
    } while (0)

static tmk_params params(int nx, int ny, double dx)
{
    tmk_params p{};
    const double cs = 3464.0, cp = 6000.0;
    p.cs = cs; p.cp = cp; p.G = 2.67e-3 * cs * cs;
    p.sxx0 = p.syy0 = p.szz0 = -120.0; p.sxy0 = 70.0;
    p.fault_kind = TMK_FAULT_SW;
    p.fs = 0.677; p.fd = 0.525; p.dw = 0.4; p.sw_rupture_thr = 1e-3;
    p.num_patches = 1; p.xc[0] = nx * dx / 2; p.xw[0] = 1500.0; p.tau_p[0] = 81.6;
    p.fric_width[0] = 1e40; p.fric_width[1] = 1e40; p.outside_f = 10.0; p.ramp_w = 1e40;
    p.normal_pred = TMK_PRED_PPM; p.fourth_order = 1; p.prim_limiting = 1;
    p.dx = dx;
    p.domain.hi[0] = nx - 1; p.domain.hi[1] = ny - 1;
    return p;
}

// ---------------------------------------------------------------------------
// register faces: every entry a hierarchy's registers read is stored by one workgroup of the launch
// ---------------------------------------------------------------------------
typedef std::map<std::pair<const double*, int>, int> Writers;

// the faces that the workgroups of a level's launch compute and store: of a tile, a strip or a boundary
// piece, the lo x faces of its cells and of the column beyond, the lo y faces of its cells and of the row
// beyond (the kernels' conditions on lx, ly)
template <typename T>
static void writers_of(const Group& G, bool all, Writers& w)
{
    const Patch<T>* pts = (const Patch<T>*)G.patches_dev[0];
    for (int q = 0; q < G.ntiles; ++q) {
        const Tile& t = G.tiles_dev[q];
        const Patch<T>& p = pts[t.patch];
        const int mw = p.vhi0 - p.vlo0 + 3;
        for (int d = 0; d < 2; ++d)
            for (int j = t.y0; j <= t.y1 + (d == 1); ++j)
                for (int i = t.x0; i <= t.x1 + (d == 0); ++i) {
                    const unsigned char* mk = p.fmask + (size_t)(i - p.vlo0 + 1) + (size_t)(j - p.vlo1 + 1) * mw;
                    const bool lo = all || (d == 0 ? i > t.x0 : j > t.y0), hi = all || (d == 0 ? i <= t.x1 : j <= t.y1);
                    if (!register_face(d == 0 ? mk[-1] : mk[-mw], *mk, lo, hi)) continue;
                    const int fnx = p.vhi0 - p.vlo0 + 1 + (d == 0);
                    ++w[{p.F[d], (i - p.vlo0) + (j - p.vlo1) * fnx}];
                }
    }
}

template <typename T>
static int registers_case(const std::vector<std::vector<tmk_box>>& boxes, int nx, int ny, int r, int march)
{
    const int prec = sizeof(T) == sizeof(double) ? TMK_PREC_FP64 : TMK_PREC_FP32_BULK;
    std::vector<tmk_ctx*> ctx;
    std::vector<tmk_level*> lev;
    int lnx = nx, lny = ny;
    double dx = 100.0;
    for (const auto& b : boxes) {
        const tmk_params p = params(lnx, lny, dx);
        tmk_ctx* c = nullptr;
        tmk_level* L = nullptr;
        EXPECT(tmk_ctx_create(&c, &p, prec) == TMK_OK);
        if (march >= 0) EXPECT(tmk_set_march(c, march) == TMK_OK);
        EXPECT(tmk_level_create(c, (int)b.size(), b.data(), &L) == TMK_OK);
        ctx.push_back(c);
        lev.push_back(L);
        lnx *= r; lny *= r; dx /= r;
    }
    tmk_amr* A = nullptr;
    EXPECT(tmk_amr_create((int)lev.size(), lev.data(), r, &A) == TMK_OK);
    EXPECT(tmk_amr_run(A, 1, 0.0, 1e-3) == TMK_OK);
    int shared = 0;
    std::vector<Writers> w(lev.size());
    for (int l = 0; l < A->nlev; ++l) {
        writers_of<T>(A->lv[l].grp, false, w[l]);
        for (const auto& f : w[l]) EXPECT(f.second == 1);
        Writers both;
        writers_of<T>(A->lv[l].grp, true, both);
        EXPECT(both.size() == w[l].size());  // no register face goes without its writer
        for (const auto& f : both) shared += f.second > 1;
    }
    for (int l = 0; l + 1 < A->nlev; ++l) {
        const AmrLevel& a = A->lv[l];
        const Patch<T>* crs = (const Patch<T>*)a.grp.patches_dev[0];
        const Patch<T>* fine = (const Patch<T>*)A->lv[l + 1].grp.patches_dev[0];
        EXPECT(a.nreg > 0);
        for (int k = 0; k < a.nreg; ++k) {
            const RegFace& f = ((const RegFace*)a.regf.p)[k];
            EXPECT(w[l].count({crs[f.cpatch].F[f.d], f.cface}) == 1);
            for (int m = 0; m < r; ++m) EXPECT(w[l + 1].count({fine[f.fpatch].F[f.d], f.fface[m]}) == 1);
        }
    }
    EXPECT(tmk_amr_destroy(A) == TMK_OK);
    for (tmk_level* L : lev) EXPECT(tmk_level_destroy(L) == TMK_OK);
    for (tmk_ctx* c : ctx) EXPECT(tmk_ctx_destroy(c) == TMK_OK);
    return shared;
}

static tmk_box box(int x0, int y0, int x1, int y1)
{
    tmk_box b;
    b.lo[0] = x0; b.lo[1] = y0; b.hi[0] = x1; b.hi[1] = y1;
    return b;
}

static void registers()
{
    const int nx = 72, ny = 40;
    const std::vector<tmk_box> whole = {box(0, 0, nx - 1, ny - 1)};
    // refined regions whose edges lie 3 coarse cells from the fault and from the other edges, inside and
    // out, at a strip's 58th column, and one that spans the domain; a third level inside one of them
    const std::vector<std::vector<tmk_box>> refined = {
        {box(12, 0, 27, 2)}, {box(12, 3, 27, 9)},         // covered below row 3, from row 3 on
        {box(3, 12, 20, 20)}, {box(0, 12, 2, 20)},        // column 3, both ways
        {box(30, 12, nx - 4, 20)}, {box(nx - 3, 12, nx - 1, 20)},
        {box(20, 20, 60, ny - 4)}, {box(20, ny - 3, 60, ny - 1)},
        {box(50, 10, 60, 20), box(61, 10, 64, 20)},
        {box(0, 0, nx - 1, 2)},
    };
    int shared = 0;
    for (int r : {2, 4})
        for (const auto& c : refined) {
            std::vector<std::vector<tmk_box>> b = {whole, {}};
            for (const tmk_box& q : c)
                b[1].push_back(box(q.lo[0] * r, q.lo[1] * r, (q.hi[0] + 1) * r - 1, (q.hi[1] + 1) * r - 1));
            for (int march : {-1, 0, 4, 63}) {
                shared += registers_case<float>(b, nx, ny, r, march);
                shared += registers_case<double>(b, nx, ny, r, march);
            }
        }
    const std::vector<std::vector<tmk_box>> three = {whole, {box(24, 0, 87, 31)}, {box(64, 0, 159, 5)}};
    shared += registers_case<float>(three, nx, ny, 2, -1);
    EXPECT(shared > 0);  // faces that two workgroups of a launch compute
}

// ---------------------------------------------------------------------------
// which calls fit the allocation-free call's scratch
// ---------------------------------------------------------------------------
// The rule the limit was set with: two copies of the state, the FP64 image of an FP32 one, the fluxes and
// the tables (a descriptor of 512 bytes, 20 bytes a tile, a scenario block of 1048), each part from a
// multiple of 256 bytes, within TMK_NOALLOC_SCRATCH_BYTES.
static void scratch_limit()
{
    for (int prec : {TMK_PREC_FP64, TMK_PREC_FP32_BULK})
        for (bool flux : {false, true}) {
            const int nx = 1000, ny = 240;
            const tmk_params p = params(nx, ny, 25.0);
            tmk_ctx* c = nullptr;
            EXPECT(tmk_ctx_create(&c, &p, prec) == TMK_OK);
            const size_t ts = prec == TMK_PREC_FP64 ? sizeof(double) : sizeof(float);
            int fits = 0, refused = 0, close = 0;
            for (int vny = 24; vny <= 200; ++vny)
                for (int vnx = 100; vnx < 900; ++vnx) {
                    const tmk_box v = box(8, 8, 8 + vnx - 1, 8 + vny - 1);
                    const tmk_box ub = box(v.lo[0] - 4, v.lo[1] - 4, v.hi[0] + 4, v.hi[1] + 4);
                    const size_t plane = (size_t)(vnx + 8) * (vny + 8), nU = plane * TMK_NCOMP;
                    const size_t n0 = (size_t)(vnx + 1) * vny * TMK_NCOMP, n1 = (size_t)vnx * (vny + 1) * TMK_NCOMP;
                    auto up = [](size_t b) { return (b + 255) / 256 * 256; };
                    size_t need = 2 * up(nU * ts) + (flux ? up((n0 + n1) * sizeof(double)) : 0);
                    if (prec != TMK_PREC_FP64) need += up(nU * sizeof(double));
                    int nint = 0;
                    const int nt = patch_tiles(v, c->P, c->bx, c->by, nullptr, 0, &nint);
                    need += 512 + up(20 * (size_t)nt) + 1048;
                    if (need + 8192 < TMK_NOALLOC_SCRATCH_BYTES || need > TMK_NOALLOC_SCRATCH_BYTES + 8192) continue;
                    const bool ok = need <= TMK_NOALLOC_SCRATCH_BYTES && nt <= 1024;
                    std::vector<double> U(nU, 0.0), F0(flux ? n0 : 0), F1(flux ? n1 : 0);
                    double mws = 0.0;
                    const int e = tmk_patch_update_state_noalloc(c, v, U.data(), ub, TMK_NCOMP, flux ? F0.data() : nullptr,
                                                                 flux ? F1.data() : nullptr, nullptr, ub, 0, 0.0, 1e-3, &mws);
                    EXPECT(e == (ok ? TMK_OK : TMK_E_SCRATCH));
                    fits += ok;
                    refused += !ok;
                    close += ok && need + 2048 > TMK_NOALLOC_SCRATCH_BYTES;
                }
            EXPECT(fits > 0 && refused > 0 && close > 0);
            EXPECT(tmk_ctx_destroy(c) == TMK_OK);
        }
}

// ---------------------------------------------------------------------------
// the allocation-free call's list: every FP64 box that fits the scratch has its strips and pieces
// ---------------------------------------------------------------------------
static void strip_lists()
{
    size_t longest = 0;
    for (int w : {1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 14, 30, 64, 130})
        for (int tall : {0, 1}) {
            // the longest box of this width that fits, in a domain of its own width and in a wider one
            for (int margin : {0, 1, 5}) {
                const int n = 47662 / (w + 2 * std::min(margin, 3)) - (margin ? 6 : 0);
                const int nx = tall ? w + 2 * margin : n + 2 * margin, ny = tall ? n + 2 * margin : w + 2 * margin;
                if (std::min(nx, ny) < 4) continue;  // the smallest domain
                const tmk_params p = params(nx, ny, 25.0);
                tmk_ctx* c = nullptr;
                EXPECT(tmk_ctx_create(&c, &p, TMK_PREC_FP64) == TMK_OK);
                const tmk_box v = tall ? box(margin, margin, margin + w - 1, margin + n - 1)
                                       : box(margin, margin, margin + n - 1, margin + w - 1);
                for (int rows : {0, 1, 4, 63}) {  // 0: the height the call chooses
                    if (rows) EXPECT(tmk_set_march(c, rows) == TMK_OK);
                    EXPECT(patch_may_march(c));
                    int nint = 0;
                    const std::vector<Tile> t = patch_strips(c, v, &nint, kNoAllocMaxStrips);
                    EXPECT(t.size() <= (size_t)kNoAllocMaxStrips);
                    longest = std::max(longest, t.size());
                    long long cells = 0;
                    for (const Tile& q : t) cells += (long long)(q.x1 - q.x0 + 1) * (q.y1 - q.y0 + 1);
                    EXPECT(cells == (long long)n * w);
                }
                EXPECT(tmk_ctx_destroy(c) == TMK_OK);
            }
        }
    EXPECT(longest > 1024);
}

// ---------------------------------------------------------------------------
// the pinned stages of downloads and drop-in calls
// ---------------------------------------------------------------------------
static void stages()
{
    g_pin_on = true;
    const int nx = 40, ny = 30;
    const tmk_params p = params(nx, ny, 25.0);
    const tmk_box v = box(0, 0, nx - 1, ny - 1), ub = box(-4, -4, nx + 3, ny + 3), bb = box(-4, 0, nx + 3, 0);
    const size_t nU = (size_t)(nx + 8) * (ny + 8) * TMK_NCOMP, nB = (size_t)(nx + 8) * TMK_NBDRY_SW;
    auto calls = [&](int dev, int precision) {
        EXPECT(hipSetDevice(dev) == hipSuccess);
        tmk_ctx* c = nullptr;
        tmk_level* L = nullptr;
        EXPECT(tmk_ctx_create(&c, &p, precision) == TMK_OK);
        EXPECT(tmk_level_create(c, 1, &v, &L) == TMK_OK);
        std::vector<double> U(nU, 0.0), B(nB, 0.0);
        double mws = 0.0;
        for (int k = 0; k < 20; ++k) {
            EXPECT(tmk_level_download(L, 0, U.data(), B.data()) == TMK_OK);
            std::fill(U.begin(), U.end(), 0.0);
            (void)tmk_patch_update_state_noalloc(c, v, U.data(), ub, TMK_NCOMP, nullptr, nullptr, B.data(), bb,
                                                 TMK_NBDRY_SW, 0.0, 1e-3, &mws);
        }
        EXPECT(tmk_level_destroy(L) == TMK_OK);
        EXPECT(tmk_ctx_destroy(c) == TMK_OK);
    };
    // ten devices from one process: each context leaves its device an idle stage, and none is made or freed again
    for (int round = 0; round < 2; ++round)
        for (int dev = 0; dev < 10; ++dev) {
            calls(dev, dev % 2 ? TMK_PREC_FP64 : TMK_PREC_FP32_BULK);
            EXPECT(stage_pool().idle[dev] != nullptr);
            EXPECT(g_pins == (round ? 10 : dev + 1) && g_frees == 0);
        }
    // forty readers of one device at once: at most STAGE_MOST stages of it, none freed
    std::vector<std::thread> th;
    std::atomic<int> ready{0};
    for (int t = 0; t < 40; ++t)
        th.emplace_back([&, t] {
            ++ready;
            while (ready < 40) std::this_thread::yield();
            calls(3, t % 2 ? TMK_PREC_FP64 : TMK_PREC_FP32_BULK);
        });
    for (std::thread& t : th) t.join();
    EXPECT(g_pins <= 9 + STAGE_MOST && g_frees == 0 && stage_pool().live[3] <= STAGE_MOST);
    // all stages of a device in use: calls copy, and pin nothing
    EXPECT(hipSetDevice(2) == hipSuccess);
    std::vector<HostStage*> held;
    while (HostStage* S = stage_take()) held.push_back(S);
    EXPECT(held.size() == (size_t)STAGE_MOST);
    const int pins = g_pins;
    calls(2, TMK_PREC_FP64);
    calls(2, TMK_PREC_FP32_BULK);
    EXPECT(g_pins == pins && g_frees == 0);
    for (HostStage* S : held) stage_give(S);
    // trimming frees the current device's, no other's
    const int before = g_pinned;
    EXPECT(tmk_cache_trim() == TMK_OK);
    EXPECT(g_pinned == before - STAGE_MOST && !stage_pool().idle[2] && stage_pool().live[2] == 0);
    EXPECT(stage_pool().idle[1] && stage_pool().idle[3]);
    for (int dev = 0; dev < 10; ++dev) {
        EXPECT(hipSetDevice(dev) == hipSuccess);
        EXPECT(tmk_cache_trim() == TMK_OK);
    }
    EXPECT(g_pinned == 0);
}

// ---------------------------------------------------------------------------
// device memory that an upload stages through
// ---------------------------------------------------------------------------
static void upload_staging()
{
    const int cases[][2] = {{50, TMK_PREC_FP64}, {50, TMK_PREC_FP32_BULK}, {210, TMK_PREC_FP32_BULK},
                            {230, TMK_PREC_FP32_BULK}, {400, TMK_PREC_FP64}, {400, TMK_PREC_FP32_BULK}};
    for (const auto& k : cases) {
        const int nx = k[0], ny = 200, prec = k[1];
        const tmk_params p = params(nx, ny, 25.0);
        const tmk_box v = box(0, 0, nx - 1, ny - 1);
        const size_t nU = (size_t)(nx + 8) * (ny + 8) * TMK_NCOMP, nB = (size_t)(nx + 8) * TMK_NBDRY_SW;
        tmk_ctx* c = nullptr;
        tmk_level* L = nullptr;
        EXPECT(tmk_ctx_create(&c, &p, prec) == TMK_OK);
        EXPECT(tmk_level_create(c, 1, &v, &L) == TMK_OK);
        std::vector<double> U(nU, 0.0), B(nB, 0.0);
        EXPECT(tmk_level_upload(L, 0, U.data(), B.data()) == TMK_OK);
        // no more than the box's planes in the level's own type, but for what fits 8 MiB
        const size_t whole = nU * sizeof(double);
        EXPECT(c->bufs[7].n == (prec == TMK_PREC_FP64 || whole <= (8u << 20) ? whole : whole / 2));
        EXPECT(tmk_level_destroy(L) == TMK_OK);
        EXPECT(tmk_ctx_destroy(c) == TMK_OK);
    }
}

// ---------------------------------------------------------------------------
// a download when host memory runs out while it starts its threads
// ---------------------------------------------------------------------------
static void reader_threads()
{
    g_pin_on = true;
    const int nx = 400, ny = 300;
    const tmk_params p = params(nx, ny, 25.0);
    const tmk_box v = box(0, 0, nx - 1, ny - 1);
    const size_t nU = (size_t)(nx + 8) * (ny + 8) * TMK_NCOMP, nB = (size_t)(nx + 8) * TMK_NBDRY_SW;
    tmk_ctx* c = nullptr;
    tmk_level* L = nullptr;
    EXPECT(tmk_ctx_create(&c, &p, TMK_PREC_FP64) == TMK_OK);
    EXPECT(tmk_level_create(c, 1, &v, &L) == TMK_OK);
    std::vector<double> U(nU), B(nB);
    for (int left : {-1, 0, 1, 2}) {
        std::fill(U.begin(), U.end(), 1.0);
        g_new_left = left;
        const int e = tmk_level_download(L, 0, U.data(), B.data());
        g_new_left = -1;
        EXPECT(e == TMK_OK);
        for (double u : U) EXPECT(u == 0.0);  // every piece was carried on (no kernel ran: the slots hold zeros)
    }
    EXPECT(tmk_level_destroy(L) == TMK_OK);
    EXPECT(tmk_ctx_destroy(c) == TMK_OK);
    EXPECT(tmk_cache_trim() == TMK_OK);
}

// ---------------------------------------------------------------------------
// strip heights: what a level reports is what its launches take, alone and in a batch
// ---------------------------------------------------------------------------
static void strip_heights()
{
    const int sizes[][2] = {{60, 40}, {261, 131}, {300, 150}, {1021, 509}, {1500, 750}, {4096, 2048}};
    for (int prec : {TMK_PREC_FP64, TMK_PREC_FP32_BULK}) {
        bool other = false;  // some level takes another height than the nominal one
        for (const auto& n : sizes) {
            const tmk_params p = params(n[0], n[1], 25.0);
            const tmk_box v = box(0, 0, n[0] - 1, n[1] - 1);
            tmk_ctx* c = nullptr;
            EXPECT(tmk_ctx_create(&c, &p, prec) == TMK_OK);
            tmk_level* L[3] = {};
            for (tmk_level*& l : L) {
                EXPECT(tmk_level_create(c, 1, &v, &l) == TMK_OK);
                if (n[0] == 4096) break;  // (one is large enough)
            }
            int rows = 0, bx = 0, by = 0, r2 = 0, x2 = 0, y2 = 0;
            EXPECT(tmk_level_get_update_shape(L[0], &rows, &bx, &by) == TMK_OK);
            EXPECT(group_build(L[0]->own, {L[0]}, {0}, 1) == TMK_OK);
            EXPECT(L[0]->own.march == rows);
            other = other || rows != 32;
            if (L[1]) {
                // the shape of one level set on another: the same launches, and the two share them; so does
                // the nominal height, and no other
                EXPECT(tmk_level_set_update_shape(L[1], rows, bx, by) == TMK_OK);
                EXPECT(tmk_level_get_update_shape(L[1], &r2, &x2, &y2) == TMK_OK);
                EXPECT(r2 == rows && x2 == bx && y2 == by);
                for (int set : {rows, 32, 20}) {
                    EXPECT(tmk_level_set_update_shape(L[2], set, bx, by) == TMK_OK);
                    for (int first : {0, 2}) {
                        tmk_batch* B = nullptr;
                        EXPECT(tmk_batch_create(&B) == TMK_OK);
                        EXPECT(tmk_batch_add(B, L[first], 0.0, 1e-3) == TMK_OK);
                        const int e = tmk_batch_add(B, L[2 - first], 0.0, 1e-3);
                        EXPECT(e == (set == 20 && rows != 20 ? TMK_E_ARG : TMK_OK));
                        EXPECT(tmk_batch_run(B, 1) == TMK_OK);
                        EXPECT(B->grp.march == (e == TMK_OK ? set : first ? set : rows));
                        EXPECT(tmk_batch_destroy(B) == TMK_OK);
                    }
                }
            }
            for (tmk_level* l : L)
                if (l) EXPECT(tmk_level_destroy(l) == TMK_OK);
            EXPECT(tmk_ctx_destroy(c) == TMK_OK);
        }
        EXPECT(other);
    }
}

// ---------------------------------------------------------------------------
// divisions in two operations: what the host decides for a divisor, and what the functions give
// ---------------------------------------------------------------------------
// stdin: lines "div B N x1 .. xN" -> "flag yh yl, then divr2(x) divr(x) each"; "par cs cp G" -> the material's
// flag, rho Zp Zs and their low words; "third N x1 .. xN" -> div3(x) div6(x) each; hexadecimal floats
static void division()
{
    char kind[16];
    while (scanf("%15s", kind) == 1) {
        if (!strcmp(kind, "div")) {
            double b;
            int n;
            EXPECT(scanf("%la %d", &b, &n) == 2);
            const double y = 1.0 / b, yl = recip_low(b, y);
            printf("%d %a %a", (int)div2_exact(b), y, yl);
            for (double x; n > 0 && scanf("%la", &x) == 1; --n) printf(" %a %a", divr2(x, y, yl), divr(x, b, y));
        } else if (!strcmp(kind, "par")) {
            tmk_params p = params(32, 32, 1.0);
            EXPECT(scanf("%la %la %la", &p.cs, &p.cp, &p.G) == 3);
            DevParams P;
            fill_dev_params(p, P);
            printf("%d %a %a %a %a %a %a", P.div2, P.rho, P.Zp, P.Zs, P.lrho, P.l2Zp, P.l2Zs);
        } else if (!strcmp(kind, "third")) {
            int n;
            EXPECT(scanf("%d", &n) == 1);
            for (double x; n > 0 && scanf("%la", &x) == 1; --n) printf("%a %a ", div3(x), div6(x));
        } else {
            fail("division: no such line", __LINE__);
        }
        printf("\n");
    }
}

int main(int argc, char** argv)
{
    const char* const what = argc > 1 ? argv[1] : "";
    if (!strcmp(what, "registers")) registers();
    else if (!strcmp(what, "scratch_limit")) scratch_limit();
    else if (!strcmp(what, "strip_lists")) strip_lists();
    else if (!strcmp(what, "stages")) stages();
    else if (!strcmp(what, "upload_staging")) upload_staging();
    else if (!strcmp(what, "reader_threads")) reader_threads();
    else if (!strcmp(what, "strip_heights")) strip_heights();
    else if (!strcmp(what, "division")) division();
    else fail("no such check", __LINE__);
    printf("%s ok\n", what);
    return 0;
}
