// CPU check of the device memory that the host code takes, keeps and gives back, on a runtime
// without a device (fake_hip.h).  Usage: memory_check <check>; prints OK or what failed.
#include "fake_hip.h"

#include "../../blochlib_amd/csrc/blfid_host.cpp"

#include <functional>

static int fails = 0;

// host allocations fail while this is set
static bool no_host_memory = false;
void *operator new(size_t n) {
    void *p = no_host_memory ? nullptr : std::malloc(n);
    if (!p) throw std::bad_alloc();
    return p;
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, size_t) noexcept { std::free(p); }
#define REQUIRE(c)                                                                               \
    do {                                                                                         \
        if (!(c)) {                                                                              \
            std::printf("FAIL line %d: %s (%s)\n", __LINE__, #c, blfid_last_error());            \
            fails++;                                                                             \
        }                                                                                        \
    } while (0)

constexpr size_t GB = (size_t)1 << 30, MB = (size_t)1 << 20;

// S protons with every dipole coupling and a shielding each
struct Sys {
    std::vector<int> iso;
    std::vector<double> csa, dip;
    blfid_system s;
    explicit Sys(int S) : iso(S, 1) {
        for (int i = 0; i < S; i++) {
            const double c[7] = {100.0 * i, 3000.0, 0.3, (double)i, 10.0 * i, 20.0, 30.0};
            csa.insert(csa.end(), c, c + 7);
            for (int j = i + 1; j < S; j++) {
                const double d[6] = {-9000.0, (double)i, (double)j, 0.0, 15.0 * j, 25.0};
                dip.insert(dip.end(), d, d + 6);
            }
        }
        s = {S, iso.data(), S, csa.data(), (int)(dip.size() / 6), dip.data(), 0, nullptr};
    }
};
// I+ of every spin, and with general set a second operator that is no (D + D^H) / 2
static std::vector<double> op(int S, bool plus, bool general = false) {
    const size_t N = (size_t)1 << S;
    std::vector<double> m(2 * N * N, 0.0);
    for (int i = 0; i < S; i++)
        for (size_t a = 0; a < N; a++)
            if (a >> i & 1) {
                const size_t b = a ^ ((size_t)1 << i);
                m[2 * (b + a * N)] = plus ? 1.0 : 0.5;
                if (!plus) m[2 * (a + b * N)] = general ? 0.25 * (i + 1) : 0.5;
            }
    return m;
}
static blfid_plan *plan(int S, int n, int npts, blfid_precision prec, int K, bool general = false) {
    Sys sy(S);
    blfid_plan *p = nullptr;
    REQUIRE(blfid_plan_create(&sy.s, 10000.0, 54.7356, 10000.0 * n, npts, 0.0, prec, &p) == BLFID_OK);
    const auto rho = op(S, false, general), det = op(S, true);
    REQUIRE(blfid_plan_set_operators(p, rho.data(), det.data()) == BLFID_OK);
    std::vector<double> a(K, 0.3), w(K, 1.0);
    REQUIRE(blfid_plan_set_powder(p, a.data(), a.data(), a.data(), w.data(), K) == BLFID_OK);
    return p;
}

// A workspace that fits the device once the memory kept from destroyed plans is given up.
static void workspace() {
    fake::limit = 4 * GB;
    blfid_plan *p = plan(6, 64, 512, BLFID_FP64, 400);
    REQUIRE(blfid_plan_run(p, 1, nullptr) == BLFID_OK);
    blfid_plan_destroy(p);
    REQUIRE(fake::used > 256 * MB); // kept
    blfid_workspace *w = nullptr;
    REQUIRE(blfid_workspace_create((double)(fake::limit - 64 * MB), &w) == BLFID_OK);
    blfid_workspace_destroy(w);
    // one beyond the device is still refused, with no error left for the next launch to report
    w = nullptr;
    REQUIRE(blfid_workspace_create((double)(fake::limit + GB), &w) == BLFID_ERR_NOMEM && !w);
    REQUIRE(hipGetLastError() == hipSuccess);
}

// Memory kept from destroyed plans and states is bounded, counted, and given back on request.
static void release() {
    fake::limit = 64 * GB;
    double kept = -1;
    REQUIRE(blfid_memory_kept(&kept) == BLFID_OK && kept == 0);
    std::vector<blfid_plan *> ps;
    for (int i = 0; i < 4; i++) {
        ps.push_back(plan(6, 64, 512, BLFID_FP64, 400));
        REQUIRE(blfid_plan_set_memory_budget(ps.back(), 3.0 * GB) == BLFID_OK);
        REQUIRE(blfid_plan_run(ps.back(), 1, nullptr) == BLFID_OK);
    }
    for (auto *p : ps) blfid_plan_destroy(p);
    REQUIRE(blfid_memory_kept(&kept) == BLFID_OK && kept > 0 && kept <= 4.0 * GB);
    REQUIRE((double)fake::used == kept); // nothing else is left of the plans
    REQUIRE(blfid_memory_release() == BLFID_OK);
    REQUIRE(blfid_memory_kept(&kept) == BLFID_OK && kept == 0 && fake::used == 0);
    blfid_plan *p = plan(3, 16, 64, BLFID_FP64, 10);
    REQUIRE(blfid_plan_run(p, 1, nullptr) == BLFID_OK);
    blfid_plan_destroy(p);
    REQUIRE(blfid_memory_kept(nullptr) == BLFID_ERR_INVALID);
}

// Kept blocks that went with a hipDeviceReset are neither handed out nor freed: their addresses
// belong to whoever allocated since.
static void reset() {
    blfid_plan_destroy(plan(4, 32, 128, BLFID_FP64, 50));
    REQUIRE(fake::used > 0);
    std::map<size_t, size_t> was;
    for (auto &kv : fake::mem) was[kv.first] = kv.second.bytes;
    fake::reset();
    // another allocator takes the same addresses in the same sizes
    std::vector<void *> other(was.size());
    size_t i = 0;
    for (auto &kv : was) REQUIRE(hipMalloc(&other[i++], kv.second) == hipSuccess);
    const auto theirs = fake::mem;
    blfid_plan *p = plan(4, 32, 128, BLFID_FP64, 50);
    REQUIRE(fake::mem.size() > theirs.size()); // blocks of its own
    blfid_plan_destroy(p);
    REQUIRE(blfid_memory_release() == BLFID_OK);
    REQUIRE(fake::mem.size() == theirs.size());
    for (auto &kv : theirs) REQUIRE(fake::mem.count(kv.first) && fake::mem[kv.first].id == kv.second.id);
    REQUIRE(hipGetLastError() == hipSuccess);
}

// A plan's and a state's working storage stay within their memory budgets, whichever block they
// come from: a kept one that is larger, or a new one whose size would be rounded up.
static void budget() {
    blfid_plan *p = plan(5, 64, 256, BLFID_FP64, 300);
    REQUIRE(blfid_plan_set_memory_budget(p, 400.0 * MB) == BLFID_OK);
    REQUIRE(blfid_plan_run(p, 1, nullptr) == BLFID_OK);
    blfid_plan_destroy(p); // keeps about 400 MB
    p = plan(5, 64, 256, BLFID_FP64, 300);
    for (double b : {390.0 * MB, 380.0 * MB + 4097, 300.0 * MB + 12345}) {
        p->own_ws.release();
        REQUIRE(blfid_plan_set_memory_budget(p, b) == BLFID_OK);
        REQUIRE(blfid_plan_run(p, 1, nullptr) == BLFID_OK);
        REQUIRE((double)p->own_ws.blk.bytes <= b);
        REQUIRE(fake::mem.at((size_t)p->own_ws.p).bytes <= b);
        p->own_ws.release();
        REQUIRE(blfid_plan_run_slice(p, 0, 300, 1, nullptr) == BLFID_OK);
        REQUIRE((double)p->own_ws.blk.bytes <= b);
        p->own_ws.release();
        REQUIRE(blfid_plan_graph_capture(p, 1) == BLFID_OK);
        REQUIRE((double)p->own_ws.blk.bytes <= b);
    }
    blfid_plan_destroy(p);
    Sys sy(5);
    std::vector<double> a(300, 0.3), dt(4, 1e-6);
    blfid_state *st = nullptr;
    REQUIRE(blfid_state_create(5, 300, a.data(), a.data(), a.data(), a.data(), &st) == BLFID_OK);
    for (double b : {3.0 * MB, 1.0 * MB + 300}) {
        st->ws.release();
        REQUIRE(blfid_state_set_memory_budget(st, b) == BLFID_OK);
        REQUIRE(blfid_state_apply(st, &sy.s, 10000.0, 54.7, 4, nullptr, dt.data(), 0, nullptr, 1, nullptr) == BLFID_OK);
        REQUIRE(fake::mem.at((size_t)st->ws.p).bytes <= b);
    }
    blfid_state_destroy(st);
}

// Setting up plans never frees memory (which waits for all work on the device): blocks that 256
// requests have passed over go with the next released plan.
static void age() {
    blfid_plan_destroy(plan(6, 64, 512, BLFID_FP64, 400));
    blfid_plan *big = plan(6, 64, 512, BLFID_FP64, 400);
    REQUIRE(blfid_plan_run(big, 1, nullptr) == BLFID_OK);
    blfid_plan_destroy(big);
    double kept = 0, now = 0;
    REQUIRE(blfid_memory_kept(&kept) == BLFID_OK && kept > 0);
    const long freed = fake::n_free, waits = fake::n_sync;
    std::vector<blfid_plan *> ps;
    for (int i = 0; i < 120; i++) ps.push_back(plan(2, 16, 64, BLFID_FP64, 10)); // three requests each
    REQUIRE(fake::n_free == freed && fake::n_sync == waits);
    blfid_plan_destroy(ps.back());
    ps.pop_back();
    REQUIRE(fake::n_free > freed);
    REQUIRE(blfid_memory_kept(&now) == BLFID_OK && now < kept / 10);
    for (auto *p : ps) blfid_plan_destroy(p);
}

// Releasing plans takes no host memory (a destructor that threw would end the process).
static void host_memory() {
    blfid_plan *p = plan(4, 32, 128, BLFID_FP64, 50);
    REQUIRE(blfid_plan_run(p, 1, nullptr) == BLFID_OK);
    no_host_memory = true;
    blfid_plan_destroy(p);
    const blfid_status st = blfid_memory_release();
    no_host_memory = false;
    REQUIRE(st == BLFID_OK && fake::used == 0);
}

// Working storage of one crystallite as earlier versions of the library laid it out, from the plan's
// own tables: full scratch-slot counts whatever the powder, eigen-solver slots of the block's matrix
// alone, FID parts of 64 correlation chunks.  `part` > 0: the slot regions cut to that many bytes.
static size_t former_need(const blfid_plan *p, double part = 0) {
    blfid_layout::Shape s = shape_of(p);
    const size_t L = s.Lsum, bm2 = (size_t)s.bmax * s.bmax, cs = s.prec ? 8 : 16, rs = s.prec ? 4 : 8;
    auto slots = [&](double total, double per, int lo, int hi) {
        const double c = std::max<double>(lo, std::min<double>(hi, std::floor(total / per)));
        return (size_t)(part > 0 ? std::max(1.0, std::min(c, std::floor(part / per))) : c);
    };
    const bool p2 = (s.n & (s.n - 1)) == 0 && s.n >= 16 && s.n <= 512;
    const int ch = p2 ? CORR_SPAN / s.n : std::max(1, std::min(CORR_SPAN / s.n, 256 / ((s.n + 7) / 8)));
    const size_t nchunk = (p->Etot + ch - 1) / ch, parts = (nchunk + 63) / 64;
    const size_t sz[] = {s.n * L * cs, s.n * L * cs, s.n * (size_t)s.Estr * cs,
                         s.rt_from_q ? 0 : s.n * (size_t)s.Estr * cs,
                         slots(2.5e9, 9.0 * bm2 * 8.0, 64, 16384) * 9 * bm2 * rs, s.prec ? L * cs : 0, L * 16,
                         s.N * (size_t)8, slots(2.5e9, 3.0 * bm2 * 16.0, 64, 16384) * 3 * bm2 * 16,
                         parts * 2 * s.npts * 8,
                         s.eig_slots ? slots(1.0e9, bm2 * 16.0, 64, 2048) * bm2 * 16 : 0,
                         blfid_layout::ngroups(s.K) * 4 * (size_t)s.npts * 8};
    size_t o = 0;
    for (size_t x : sz) o += blfid_layout::align256(x);
    return o;
}
// What fitted a memory budget, a workspace or the static scratch before still does.
static void accepted() {
    fake::limit = (size_t)256 << 30;
    const struct { int S, n, npts; blfid_precision prec; int K; bool general; } cases[] = {
        {5, 64, 512, BLFID_C64, 2000, false},     {6, 128, 2048, BLFID_C64, 1000, true},
        {8, 128, 2048, BLFID_C64, 500, true},     {9, 32, 256, BLFID_C64, 1000, false},
        {9, 32, 256, BLFID_FP64, 1000, true},     {10, 16, 64, BLFID_C64, 500, false},
        {6, 64, 300000, BLFID_C64, 200, true},    {6, 45, 2000000, BLFID_FP64, 100, true},
        {7, 100, 1000000, BLFID_C64, 300, false},
    };
    for (auto &c : cases) {
        blfid_plan *p = plan(c.S, c.n, c.npts, c.prec, c.K, c.general);
        const double need = (double)former_need(p);
        REQUIRE(blfid_plan_set_memory_budget(p, need) == BLFID_OK);
        REQUIRE(blfid_plan_run(p, 1, nullptr) == BLFID_OK);
        REQUIRE((double)p->own_ws.blk.bytes <= need);
        p->own_ws.release();
        for (int k = 0; k < 3; k++) REQUIRE(blfid_plan_run_slice(p, k * c.K / 3, (k + 1) * c.K / 3, 1, nullptr) == BLFID_OK);
        REQUIRE((double)p->own_ws.blk.bytes <= need);
        p->own_ws.release();
        REQUIRE(blfid_plan_graph_capture(p, 1) == BLFID_OK);
        blfid_workspace *w = nullptr;
        REQUIRE(blfid_workspace_create(need, &w) == BLFID_OK);
        REQUIRE(blfid_plan_set_workspace(p, w) == BLFID_OK);
        REQUIRE(blfid_plan_run(p, 1, nullptr) == BLFID_OK);
        REQUIRE(blfid_plan_set_workspace(p, nullptr) == BLFID_OK);
        blfid_workspace_destroy(w);
        double out = 0;
        if (former_need(p, BLFID_NOALLOC_SCRATCH_BYTES / 8.0) <= BLFID_NOALLOC_SCRATCH_BYTES)
            REQUIRE(blfid_plan_run_noalloc(p, 1, &out, nullptr) == BLFID_OK);
        blfid_plan_destroy(p);
    }
}

// Hand-overs and fetches copy in pieces of more than 16 KiB that fit the pinned buffer, whatever the
// size of the plan's tables and of its FID.
static void copies() {
    fake::limit = (size_t)256 << 30;
    for (int S : {1, 3, 10})
        for (int npts : {1, 64, 1039, 1040, 1041, 5000, 400000}) {
            blfid_plan *p = plan(S, 16, npts, BLFID_FP64, S == 3 ? 200000 : 7, true);
            REQUIRE(blfid_plan_run(p, 1, nullptr) == BLFID_OK);
            std::vector<double> fid(2 * npts + 1, 1.5);
            REQUIRE(blfid_plan_fetch(p, fid.data()) == BLFID_OK);
            REQUIRE(fid[2 * npts] == 1.5 && fid[2 * npts - 1] == 0.0); // the whole FID and no more
            REQUIRE(p->fid_out.blk.bytes >= std::max((size_t)16 * npts, COPY_LEAST));
            blfid_plan_destroy(p);
            if (S == 10 && npts > 1) break;
        }
    REQUIRE(fake::copy_min > 16 * 1024 && fake::copy_max <= COPY_PIECE);
}

// The fixed storage that blfid_plan_stats names is that of any powder: a budget made from it for a
// batch of crystallites holds the batch after the plan is given a larger powder.
static void footprint() {
    fake::limit = (size_t)256 << 30;
    for (auto prec : {BLFID_FP64, BLFID_C64})
        for (int S : {5, 8, 9}) {
            blfid_plan *p = plan(S, 32, 256, prec, 10);
            double st[6];
            REQUIRE(blfid_plan_stats(p, st) == BLFID_OK);
            const double budget = st[5] + 64 * st[4];
            const size_t group = blfid_layout::ngroups(3000) * 4 * 256 * 8 / (size_t)st[4] + 1;
            std::vector<double> a(3000, 0.3);
            REQUIRE(blfid_plan_set_powder(p, a.data(), a.data(), a.data(), a.data(), 3000) == BLFID_OK);
            REQUIRE(blfid_plan_set_memory_budget(p, budget) == BLFID_OK);
            REQUIRE(blfid_plan_run(p, 1, nullptr) == BLFID_OK);
            REQUIRE(p->Kb + (int)group >= 64);
            blfid_plan_destroy(p);
        }
}

// Steps per period beyond what the correlation kernel holds on chip are refused, the most it holds
// are not.
static void steps() {
    Sys sy(2);
    blfid_plan *p = nullptr;
    for (int n : {2049, 3000, 100000}) {
        REQUIRE(blfid_plan_create(&sy.s, 10.0, 54.7356, 10.0 * n, 64, 0.0, BLFID_FP64, &p) == BLFID_ERR_UNSUPPORTED && !p);
        REQUIRE(corr_chunk(n) * (long)n > CORR_SPAN);
    }
    for (int n = 1; n <= 2048; n++) {
        REQUIRE(corr_use_fft(n) || corr_chunk(n) * n <= CORR_SPAN);
        REQUIRE(corr_use_fft(n) || corr_chunk(n) * ((n + CORR_PPT - 1) / CORR_PPT) <= 256);
    }
    REQUIRE(blfid_plan_create(&sy.s, 10.0, 54.7356, 10.0 * 2048, 64, 0.0, BLFID_FP64, &p) == BLFID_OK);
    blfid_plan_destroy(p);
}

int main(int argc, char **argv) {
    const std::map<std::string, std::function<void()>> checks = {{"workspace", workspace}, {"release", release}, {"reset", reset}, {"budget", budget}, {"age", age}, {"host_memory", host_memory}, {"accepted", accepted}, {"copies", copies}, {"footprint", footprint}, {"steps", steps}};
    std::setvbuf(stdout, nullptr, _IONBF, 0);
    if (argc != 2 || !checks.count(argv[1])) return 2;
    checks.at(argv[1])();
    if (!fails) std::printf("OK\n");
    return fails ? 1 : 0;
}
