// Checks of the library's device and pinned memory on a HIP runtime of host memory (fake_hip.h): the
// name of a check is the argument; exit status 0 when it holds.
#include "fake_hip.h"
#include "hv_internal.h"
#include <unistd.h>
#include <memory>
#include <string>
#include <thread>

#define CHECK(c)                                                            \
    do {                                                                    \
        if (!(c)) {                                                         \
            std::printf("%s:%d: %s\n", __FILE__, __LINE__, #c);             \
            return 1;                                                       \
        }                                                                   \
    } while (0)

constexpr size_t MiB = (size_t)1 << 20;

// Work queued for an export that fails part way is waited for before its buffer is another's.
static int failed_export() {
    const int nv = 1000, D = 3;
    hv_mesh m;
    m.D = D;
    m.N = 200;
    m.nreal = 200;
    m.nv = nv;
    std::vector<int> ids(nv), key(nv * (D + 1));
    std::vector<double> x(nv * D);
    for (int v = 0; v < nv; ++v) ids[v] = v;
    m.ids.p = ids.data();
    m.key.p = key.data();
    m.x.p = x.data();
    std::vector<int64_t> sig(nv * (D + 1));
    std::vector<double> coords(nv * D);
    CHECK(hv_mesh_export(&m, sig.data(), coords.data()) == HV_OK);
    const int all = fake::S().launches;
    CHECK(all > 2);
    for (int k = 0; k < all; ++k) {
        fake::S().launches = 0;
        fake::S().fail_at = k;
        CHECK(hv_mesh_export(&m, sig.data(), coords.data()) == HV_ERR_DEVICE);
        CHECK(fake::waiting() == 0);
    }
    return 0;
}

// The same of the objects themselves, when their owner leaves before it has waited; one that was
// settled does not touch its stream again.
static int queued_work() {
    hipStream_t st = nullptr;
    CHECK(hipStreamCreateWithFlags(&st, 0) == hipSuccess);
    {
        HvScratch b(0, 1000, st);
        fake::queue(st);
    }
    CHECK(fake::waiting() == 0);
    {
        HvPinned b(st);
        fake::queue(st);
    }
    CHECK(fake::waiting() == 0);
    {
        HvScratch b(0, 1000, st);
        HvPinned q(st);
        b.settled();
        q.settled();
        fake::queue(st);
    }
    CHECK(fake::waiting() == 1);
    return 0;
}

// An object released at the end of the process, after the library's own statics are gone: the handler
// is registered before any library is initialised, so it runs last.
static HvScratch* late_scratch = nullptr;
static HvPinned* late_pinned = nullptr;
extern "C" int __cxa_atexit(void (*)(void*), void*, void*) noexcept;
static void late(void*) {
    delete late_scratch;
    delete late_pinned;
    if (late_scratch) {
        HvScratch again(0, 3000, nullptr);
        HvPinned word(nullptr);
        if (!again.p || !word.p || fake::S().device.size() != 2) _exit(1);   // both taken from the stores again
    }
}
static void before_all() { __cxa_atexit(late, nullptr, nullptr); }
__attribute__((section(".preinit_array"), used)) static void (*preinit)() = before_all;
static int released_at_exit() {
    HvScratch* a = new HvScratch(0, 1000000, nullptr);
    { HvScratch b(0, 1000, nullptr); }
    late_pinned = new HvPinned(nullptr);
    { HvPinned b(nullptr); }
    late_scratch = a;
    return 0;
}

// an integral of n cells and `rows` rows, each value told by its place, and whether its export is that
static hv_integral* integral(int device, int64_t n, int64_t rows) {
    (void)hipSetDevice(device);
    hv_integral* I = new hv_integral();
    I->N = n;
    I->rows = rows;
    I->device = device;
    I->ptr = 8 * n;
    I->nbr = I->ptr + 8 * (n + 1);
    I->area = I->nbr + 8 * rows;
    I->bytes = I->area + 8 * rows;
    I->dev.reset(new HvScratch(device, I->bytes, nullptr));
    I->dev->settled();
    I->base = (char*)I->dev->p;
    for (size_t k = 0; k < I->bytes / 8; ++k) ((int64_t*)I->base)[k] = 1000 + (int64_t)k;
    return I;
}
static bool integral_intact(const hv_integral* I) {
    const int64_t n = I->N, rows = I->rows;
    std::vector<int64_t> v(2 * n + 1 + 2 * rows);   // the four arrays one after another
    if (hv_integral_export(I, (double*)v.data(), v.data() + n, v.data() + 2 * n + 1, (double*)(v.data() + 2 * n + 1 + rows),
                           nullptr) != HV_OK)
        return false;
    for (size_t k = 0; k < v.size(); ++k)
        if (v[k] != 1000 + (int64_t)k) return false;
    return true;
}

// Copies, the pinned block and an integral's export work on their own device, whichever the thread used last.
static int devices() {
    std::vector<char> a(4 * MiB, 1), b(4 * MiB, 0);
    const HvCopy one{b.data(), a.data(), a.size()};
    CHECK(hipSetDevice(0) == hipSuccess);
    CHECK(hv_copies(1, true, &one, 1) == hipSuccess && a == b);
    CHECK(fake::S().stream_device.size() > 1 && !fake::S().host.empty());
    for (auto& kv : fake::S().stream_device) CHECK(kv.second == 1);
    for (auto& kv : fake::S().host) CHECK(kv.second.device == 1);
    for (int d : fake::S().copy_device) CHECK(d == 1);
    CHECK(hipSetDevice(1) == hipSuccess);
    {
        HvLease L(0);
        CHECK(L.base && fake::S().host[L.base].device == 0);
    }
    CHECK(hipSetDevice(1) == hipSuccess);
    hv_integral* I = integral(1, 5, 20);
    CHECK(hipSetDevice(0) == hipSuccess);
    fake::S().copy_device.clear();
    CHECK(integral_intact(I));
    CHECK(!fake::S().copy_device.empty());
    for (int d : fake::S().copy_device) CHECK(d == 1);
    CHECK(hv_integral_free(I) == HV_OK);
    return 0;
}

// What is kept of destroyed objects is given back when an allocation finds no room: a pool's (grown and
// reserved), a context's points, a buffer of the store.
static int idle_given_back() {
    auto& used = fake::S().used[0];
    auto keep = []() -> int {   // 12 MiB in the store and 10 of a context, all of it idle
        { HvScratch a(0, 12 * MiB, nullptr); }
        hv_ctx* c = nullptr;
        CHECK(hv_create(&c, 0) == HV_OK);
        CHECK(c->pool->get("x", 8 * MiB));
        CHECK(hv_destroy(c) == HV_OK);
        return 0;
    };
    fake::S().limit[0] = 30 * MiB;
    for (int way = 0; way < 4; ++way) {
        hv_ctx *c = nullptr, *d = nullptr;
        CHECK(hv_create(&c, 0) == HV_OK);
        CHECK(hv_create(&d, 0) == HV_OK);
        CHECK(keep() == 0 && used >= 22 * MiB);
        std::vector<double> x(2 * 20 * MiB / 16, 0.5);
        if (way == 0) CHECK(c->pool->get("y", 20 * MiB));
        if (way == 1) CHECK(c->pool->reserve("y", 20 * MiB, c->stream));
        if (way == 2) CHECK(hv_set_points(c, 2, (int64_t)x.size() / 2, x.data()) == HV_OK);
        if (way == 3) {
            HvScratch s(0, 20 * MiB, nullptr);
            CHECK(s.p);
        }
        CHECK(!c->pool->get("z", 64 * MiB));   // more than there is: refused, and nothing lost
        hv_destroy(c);
        hv_destroy(d);
        CHECK(hv_batch_release(0) == HV_OK && used == 0);
    }
    return 0;
}

// Finished integrals make room for an allocation that finds none, and keep their results; one of another
// device stays where it is.
static int integrals_make_room() {
    fake::S().limit[0] = 30 * MiB;
    hv_integral *a = integral(0, 1000, 600000), *b = integral(0, 1000, 600000), *other = integral(1, 10, 600000);   // 9.6 MB each
    for (hv_integral* I : {a, b, other}) hv_integral_keep(I);
    CHECK(hipSetDevice(0) == hipSuccess);
    DevPool pool;
    CHECK(pool.get("y", 20 * MiB));
    CHECK(!a->dev && !b->dev && other->dev);
    CHECK(integral_intact(a) && integral_intact(b) && integral_intact(other));
    CHECK(hipSetDevice(0) == hipSuccess);
    CHECK(!pool.get("z", 64 * MiB));
    for (hv_integral* I : {a, b, other}) CHECK(hv_integral_free(I) == HV_OK);
    hv_integrals_to_host(0);   // none is left
    return 0;
}

// A thread that finds the staging taken copies all the same, and gets no lease.
static int staging_taken() {
    HvLease held(0);
    CHECK(held.base);
    int bad = 0;
    std::thread other([&]() {
        HvLease second(0);
        std::vector<char> a(4 * MiB, 3), b(4 * MiB, 0);
        const HvCopy one{b.data(), a.data(), a.size()};
        bad = second.base != nullptr || hv_copies(0, false, &one, 1) != hipSuccess || a != b;
    });
    other.join();
    CHECK(bad == 0 && fake::waiting() == 0);
    return 0;
}

int main(int argc, char** argv) {
    const std::string what = argc > 1 ? argv[1] : "";
    if (what == "devices") return devices();
    if (what == "failed_export") return failed_export();
    if (what == "staging_taken") return staging_taken();
    if (what == "integrals_make_room") return integrals_make_room();
    if (what == "idle_given_back") return idle_given_back();
    if (what == "released_at_exit") return released_at_exit();
    if (what == "queued_work") return queued_work();
    std::printf("no check of that name\n");
    return 2;
}
