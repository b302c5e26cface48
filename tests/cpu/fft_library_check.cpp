// fft_library.h against a rocFFT and a HIP runtime of which any one call fails: a failed make()
// leaves nothing behind and not ready, the next one starts again and, once it succeeds, every
// execution has an info with the caller's stream and the work buffer.
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "fft_library.h"

static int calls, fail_at, live;
static bool broken() { return ++calls == fail_at; }
struct rocfft_plan_t { int inverse; };
struct rocfft_plan_description_t { std::vector<size_t> in, out; };
static std::vector<size_t> layout[2];      // strides and distances of the last plans, in then out
struct rocfft_execution_info_t { void *stream, *work; size_t size; };
static rocfft_execution_info_t *last_info;

extern "C" {
rocfft_status rocfft_plan_create(rocfft_plan *p, rocfft_result_placement, rocfft_transform_type t, rocfft_precision,
                                 size_t, const size_t *, size_t, const rocfft_plan_description d)
{
    if (broken()) return rocfft_status_failure;
    ++live;
    *p = new rocfft_plan_t{t == rocfft_transform_type_real_inverse};
    std::vector<size_t> &v = layout[(*p)->inverse];
    v.clear();
    if (d) {
        v = d->in;
        v.insert(v.end(), d->out.begin(), d->out.end());
    }
    return rocfft_status_success;
}
rocfft_status rocfft_plan_description_create(rocfft_plan_description *d)
{
    if (broken()) return rocfft_status_failure;
    ++live;
    *d = new rocfft_plan_description_t;
    return rocfft_status_success;
}
rocfft_status rocfft_plan_description_destroy(rocfft_plan_description d) { --live; delete d; return rocfft_status_success; }
rocfft_status rocfft_plan_description_set_data_layout(rocfft_plan_description d, rocfft_array_type a, rocfft_array_type b,
                                                      const size_t *, const size_t *, size_t ni, const size_t *si,
                                                      size_t di, size_t no, const size_t *so, size_t dn)
{
    if (broken() || a == b) return rocfft_status_failure;
    d->in.assign(si, si + ni);
    d->in.push_back(di);
    d->out.assign(so, so + no);
    d->out.push_back(dn);
    return rocfft_status_success;
}
rocfft_status rocfft_plan_destroy(rocfft_plan p) { --live; delete p; return rocfft_status_success; }
rocfft_status rocfft_plan_get_work_buffer_size(const rocfft_plan p, size_t *n)
{
    *n = p->inverse ? 512 : 256;
    return broken() ? rocfft_status_failure : rocfft_status_success;
}
rocfft_status rocfft_execution_info_create(rocfft_execution_info *i)
{
    if (broken()) return rocfft_status_failure;
    ++live;
    *i = new rocfft_execution_info_t{nullptr, nullptr, 0};
    return rocfft_status_success;
}
rocfft_status rocfft_execution_info_destroy(rocfft_execution_info i) { --live; delete i; return rocfft_status_success; }
rocfft_status rocfft_execution_info_set_stream(rocfft_execution_info i, void *s)
{
    i->stream = s;
    return broken() ? rocfft_status_failure : rocfft_status_success;
}
rocfft_status rocfft_execution_info_set_work_buffer(rocfft_execution_info i, void *w, size_t n)
{
    i->work = w;
    i->size = n;
    return broken() ? rocfft_status_failure : rocfft_status_success;
}
rocfft_status rocfft_execute(const rocfft_plan, void **, void **, rocfft_execution_info i)
{
    last_info = i;
    return rocfft_status_success;
}
hipError_t hipMalloc(void **p, size_t n)
{
    if (broken()) return hipErrorOutOfMemory;
    ++live;
    *p = malloc(n);
    return hipSuccess;
}
hipError_t hipFree(void *p) { --live; free(p); return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
}

#define CHECK(x) do { if (!(x)) { printf("call %d fails: %s\n", fail_at, #x); return 1; } } while (0)

static int check(size_t pitch)
{
    const size_t n[3] = {5, 4, 3};
    const hipStream_t stream = reinterpret_cast<hipStream_t>(0x10);
    fail_at = calls = 0;
    int steps;
    {
        FftLibrary f;
        CHECK(!f.make(3, n, pitch, 11, stream));
        steps = calls;
        f.release();
    }
    for (fail_at = 1; fail_at <= steps; ++fail_at) {
        calls = 0;
        FftLibrary f;
        CHECK(f.make(3, n, pitch, 11, stream) && !f.ready() && live == 0);
        const int made = calls;
        CHECK(!f.make(3, n, pitch, 11, stream) && f.ready());       // all of it again
        CHECK(calls == made + steps);
        for (int inverse = 0; inverse < 2; ++inverse) {
            last_info = nullptr;
            CHECK(!(inverse ? f.inverse(nullptr, nullptr) : f.forward(nullptr, nullptr)));
            CHECK(last_info && last_info->stream == stream && last_info->work && last_info->size == 512);
        }
        const int before = calls;
        CHECK(!f.make(3, n, pitch, 11, stream) && calls == before); // made once
        f.release();
        CHECK(live == 0);
    }
    return 0;
}

int main()
{
    if (check(5)) return 1;
    CHECK(layout[0].empty() && layout[1].empty());                  // dense rows: rocFFT's own layout
    if (check(8)) return 1;
    CHECK((layout[0] == std::vector<size_t>{1, 8, 32, 96, 1, 3, 12, 36}));
    CHECK((layout[1] == std::vector<size_t>{1, 3, 12, 36, 1, 8, 32, 96}));
    printf("ok\n");
    return 0;
}
