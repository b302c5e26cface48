// Forward and inverse real-to-complex transforms of the grids by rocFFT, with all that an execution
// needs: both plans, their execution infos on the context's stream and one work buffer for the two.
// lengths[0] is the fastest; the rows of the real grids are pitch floats apart, everything else is dense.
#pragma once
#include <hip/hip_runtime_api.h>
#include <rocfft/rocfft.h>

#include <algorithm>
#include <cstddef>

struct FftLibrary {
    // Makes everything or nothing: a failed call leaves no plan, info or memory behind, ready() stays
    // false and a later call starts again, so no execution ever runs without the context's stream
    // (on the default stream, unordered with it).  Returns null, or what failed.
    const char *make(size_t dims, const size_t *lengths, size_t pitch, size_t batch, hipStream_t stream)
    {
        if (ready_) return nullptr;
        const char *failed = try_make(dims, lengths, pitch, batch, stream);
        if (failed) release();
        else ready_ = true;
        return failed;
    }
    bool ready() const { return ready_; }

    const char *forward(void *grid, void *spec) { return execute(fwd_, info_fwd_, grid, spec); }
    const char *inverse(void *spec, void *grid) { return execute(inv_, info_inv_, spec, grid); }

    void release()
    {
        for (rocfft_execution_info *i : {&info_fwd_, &info_inv_}) {
            if (*i) rocfft_execution_info_destroy(*i);
            *i = nullptr;
        }
        for (rocfft_plan *p : {&fwd_, &inv_}) {
            if (*p) rocfft_plan_destroy(*p);
            *p = nullptr;
        }
        if (work_) (void)hipFree(work_);
        work_ = nullptr;
        ready_ = false;
    }

private:
    const char *try_make(size_t dims, const size_t *lengths, size_t pitch, size_t batch, hipStream_t stream)
    {
        auto ok = [](rocfft_status s) { return s == rocfft_status_success; };
        for (const bool inverse : {false, true}) {
            rocfft_plan_description layout = nullptr;
            if (pitch != lengths[0]) {
                size_t real[3] = {1, 1, 1}, half[3] = {1, 1, 1}, real_size = pitch, half_size = lengths[0] / 2 + 1;
                for (size_t d = 1; d < dims; ++d) {
                    real[d] = real_size;
                    half[d] = half_size;
                    real_size *= lengths[d];
                    half_size *= lengths[d];
                }
                const rocfft_array_type r = rocfft_array_type_real, h = rocfft_array_type_hermitian_interleaved;
                const bool described =
                    ok(rocfft_plan_description_create(&layout)) &&
                    ok(rocfft_plan_description_set_data_layout(
                        layout, inverse ? h : r, inverse ? r : h, nullptr, nullptr, dims, inverse ? half : real,
                        inverse ? half_size : real_size, dims, inverse ? real : half, inverse ? real_size : half_size));
                if (!described) {
                    if (layout) rocfft_plan_description_destroy(layout);
                    return "rocfft_plan_description failed";
                }
            }
            const bool made = ok(rocfft_plan_create(
                inverse ? &inv_ : &fwd_, rocfft_placement_notinplace,
                inverse ? rocfft_transform_type_real_inverse : rocfft_transform_type_real_forward,
                rocfft_precision_single, dims, lengths, batch, layout));
            if (layout) rocfft_plan_description_destroy(layout);
            if (!made) return "rocfft_plan_create failed";
        }
        size_t w1 = 0, w2 = 0;
        if (!ok(rocfft_plan_get_work_buffer_size(fwd_, &w1)) || !ok(rocfft_plan_get_work_buffer_size(inv_, &w2)))
            return "rocfft_plan_get_work_buffer_size failed";
        const size_t size = std::max(w1, w2);
        if (size && hipMalloc(&work_, size) != hipSuccess) {
            work_ = nullptr;
            (void)hipGetLastError();
            return "no memory for rocFFT's work buffer";
        }
        for (rocfft_execution_info *i : {&info_fwd_, &info_inv_})
            if (!ok(rocfft_execution_info_create(i)) || !ok(rocfft_execution_info_set_stream(*i, stream)) ||
                (size && !ok(rocfft_execution_info_set_work_buffer(*i, work_, size))))
                return "rocfft_execution_info failed";
        return nullptr;
    }

    static const char *execute(rocfft_plan plan, rocfft_execution_info info, void *in, void *out)
    {
        void *i[1] = {in}, *o[1] = {out};
        return rocfft_execute(plan, i, o, info) == rocfft_status_success ? nullptr : "rocfft_execute failed";
    }

    rocfft_plan fwd_ = nullptr, inv_ = nullptr;
    rocfft_execution_info info_fwd_ = nullptr, info_inv_ = nullptr;
    void *work_ = nullptr;
    bool ready_ = false;
};
