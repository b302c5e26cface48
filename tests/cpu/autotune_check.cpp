// autotune.cpp on the host: the products it times are replaced by counters, HIP events by a clock
// that gives every product the time the test wants, and any product may fail.
#include <cstdio>
#include <cstdlib>
#include <map>
#include <vector>

// what fsd_internal.h needs of the device compiler
struct Dim { int x; };
static Dim threadIdx;
static inline void __syncthreads() {}
static inline int __builtin_amdgcn_update_dpp(int, int, int, int, int, bool) { return 0; }

#include "autotune.cpp"

static float now_us;
static std::vector<fsd_tuning> seen;       // knobs of every product, in order
static int product, fail_product;
static float (*cost)(const fsd_tuning &, int parts);

int k_mobility(fsd_ctx *ctx, const float4 *, const float *, float *, int parts, const float *,
               const std::function<int(bool *)> *)
{
    if (++product == fail_product) { ctx->err = "planted"; return FSD_E_HIP; }
    seen.push_back(ctx->tune);
    now_us += cost(ctx->tune, parts);
    return 0;
}
int k_rfu_apply(fsd_ctx *ctx, const float *, float *, const float *, float)
{
    if (++product == fail_product) { ctx->err = "planted"; return FSD_E_HIP; }
    now_us += ctx->tune.rfu_g == 16 ? 2.f : 3.f;
    return 0;
}
static bool no_plans, in_lds;
bool real_table_in_lds(const fsd_ctx *) { return in_lds; }
int fft_plans_3d(fsd_ctx *) { return no_plans ? FSD_E_HIP : 0; }
int k_fill(fsd_ctx *, int64_t, float, float *) { return 0; }

struct ihipEvent_t { float at; };
extern "C" {
hipError_t hipMalloc(void **p, size_t n) { *p = malloc(n); return hipSuccess; }
hipError_t hipFree(void *p) { free(p); return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { *e = new ihipEvent_t{0.f}; return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { delete e; return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) { e->at = now_us; return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t a, hipEvent_t b) { *ms = (b->at - a->at) / 1000.f; return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return ""; }
}

#define CHECK(x) do { if (!(x)) { printf("product %d fails: %s\n", fail_product, #x); return 1; } } while (0)

static bool same(const fsd_tuning &a, const fsd_tuning &b)
{
    return a.spread == b.spread && a.contract == b.contract && a.xpass == b.xpass && a.real_g == b.real_g &&
           a.real_blk == b.real_blk && a.rfu_g == b.rfu_g && a.rfu_blk == b.rfu_blk && a.tuned == b.tuned;
}

static fsd_ctx *context()
{
    fsd_ctx *ctx = new fsd_ctx();
    ctx->N = 100;
    ctx->pse.P = 6;
    ctx->tile = 8;
    ctx->contract_lds = 1;
    ctx->fft_x = true;
    return ctx;
}

int main()
{
    // every alternative slower but four lanes: the search keeps the defaults and those
    cost = [](const fsd_tuning &t, int parts) {
        return parts == 2 ? 10.f + t.spread + t.contract + t.xpass : 10.f + t.real_g + (t.real_blk == 128);
    };
    fsd_ctx *ctx = context();
    CHECK(autotune_run(ctx, nullptr) == 0);
    fsd_tuning want;
    want.real_g = 4; want.rfu_g = 16; want.rfu_blk = 128; want.tuned = 1;
    CHECK(same(ctx->tune, want));
    const int products = product;
    // a failure leaves the shapes that were set before the search
    for (fail_product = 1; fail_product <= products; ++fail_product) {
        product = 0;
        fsd_ctx *c = context();
        c->tune.contract = 1;
        const fsd_tuning before = c->tune;
        CHECK(autotune_run(c, nullptr) == FSD_E_HIP && c->err == "planted");
        CHECK(same(c->tune, before));
        delete c;
    }
    // where the workgroup size is not a choice, every lane count is timed once and the size stays
    fail_product = product = 0;
    in_lds = true;
    cost = [](const fsd_tuning &t, int) { return 10.f + t.real_g - (t.real_blk == 128); };
    ctx = context();
    CHECK(autotune_run(ctx, nullptr) == 0 && ctx->tune.real_g == 4 && ctx->tune.real_blk == 256);
    CHECK(product == products - 3 * 7);
    // without the library's plans the transforms in LDS stay, untimed against them
    fail_product = 0;
    no_plans = true;
    seen.clear();
    cost = [](const fsd_tuning &t, int) { return t.xpass ? 1.f : 10.f; };
    ctx = context();
    CHECK(autotune_run(ctx, nullptr) == 0 && ctx->tune.xpass == 0);
    for (const fsd_tuning &t : seen) CHECK(t.xpass == 0);
    printf("ok\n");
    return 0;
}
