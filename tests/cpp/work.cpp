/* The kept workspace (vt_work.h) on a device of limited memory. */
#include "vt_work.h"

#include <cstdio>
#include <cstdlib>
#include <map>

static std::map<void*, size_t> held_;
static size_t total_ = 0, limit_ = 0;
static int syncs_ = 0;
hipError_t hipMalloc(void** p, size_t bytes)
{
    if (total_ + bytes > limit_) return *p = nullptr, hipErrorUnknown;
    *p = std::malloc(16);
    held_[*p] = bytes;
    total_ += bytes;
    return hipSuccess;
}
hipError_t hipFree(void* p)
{
    if (!p) return hipSuccess;
    if (!held_.count(p)) std::abort();
    total_ -= held_[p];
    held_.erase(p);
    std::free(p);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return ++syncs_, hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }

static int bad_ = 0;
#define CHECK(x) do { if (!(x)) { ++bad_; std::printf("line %d: %s\n", __LINE__, #x); } } while (0)

int main()
{
    constexpr size_t M = 1u << 20;
    vt::DeviceWork w;
    limit_ = 1000 * M;
    {
        vt::WorkSpace a(w, nullptr);
        CHECK(a.take(100 * M) == hipSuccess && a.p());
        a.waited();
    }
    CHECK(total_ == 100 * M && syncs_ == 0);               /* kept */
    {
        vt::WorkSpace a(w, nullptr), b(w, nullptr), c(w, nullptr);
        CHECK(a.take(50 * M) == hipSuccess && total_ == 100 * M);
        CHECK(b.take(60 * M) == hipSuccess && b.p() != a.p() && total_ == 160 * M);   /* in use: its own */
        CHECK(c.take(300 * M) == hipSuccess && total_ == 460 * M);                    /* too large to keep */
        void* q = nullptr;
        CHECK(w.alloc(&q, 600 * M) != hipSuccess);         /* nothing to give back while a call uses it */
        CHECK(w.alloc(&q, 500 * M) == hipSuccess);
        hipFree(q);
        a.waited();
    }
    CHECK(total_ == 100 * M && syncs_ == 2);               /* b and c returned early */
    {
        vt::WorkSpace a(w, nullptr);
        CHECK(a.take(250 * M) == hipSuccess && total_ == 250 * M);
        a.waited();
    }
    void* q = nullptr;
    CHECK(w.alloc(&q, 900 * M) == hipSuccess && total_ == 900 * M);   /* the kept buffer makes room */
    {
        vt::WorkSpace a(w, nullptr);
        CHECK(a.take(200 * M) != hipSuccess && !a.p());
        vt::WorkSpace b(w, nullptr);
        CHECK(b.take(90 * M) == hipSuccess && b.p());
    }
    CHECK(w.give_back() && total_ == 900 * M);
    CHECK(!w.give_back());
    hipFree(q);
    CHECK(total_ == 0);
    std::printf("bad %d\n", bad_);
    return bad_;
}
