// One restore call from a prepared program: fills the call buffer's host image, uploads it and enqueues
// the call's launches, so that a call whose geometry recurs costs one entry instead of a dozen array
// operations and an entry per launch.  The host time of a call bounds restores below about 60 us of device
// work: a K+V call of one 390-token, 12-head chunk takes the host 40 us (67 with the rows filled by numpy
// and every launch entered from Python), a seven-chunk history layer 61 us (89).
#include <cstddef>
#include <cstring>

#include "common.h"

namespace rch {
namespace {

// Index of a field of an all-int64 descriptor.
#define RCH_COLUMN(type, field) static_cast<int>(offsetof(type, field) / sizeof(int64_t))

constexpr int kJobColumns = sizeof(rch_job) / 8;
constexpr int kPackColumns = sizeof(rch_pack) / 8;

const int64_t* words(int64_t address) { return reinterpret_cast<const int64_t*>(address); }

int check_call(const rch_call* call, const void* image, const void* buffer, const int64_t* jobs) {
    if (!call || !image || !buffer || !jobs || call->n_jobs <= 0 || call->n_rows < call->n_jobs ||
        call->image_bytes <= 0 || call->desc_offset < 0 ||
        call->desc_offset + call->n_rows * static_cast<int64_t>(sizeof(rch_job)) > call->image_bytes ||
        call->n_packs < 0 || call->n_launches <= 0 || !call->template_ptr || !call->rows_ptr || !call->relative_ptr ||
        !call->launches_ptr || (call->n_packs > 0 && (!call->packs_ptr || !call->packs_relative_ptr || !call->members_ptr)))
        return fail(RCH_E_CONFIG, "rch_call_run: invalid call program");
    return RCH_OK;
}

}  // namespace
}  // namespace rch

using namespace rch;

extern "C" {

int rch_call_size(void) { return static_cast<int>(sizeof(rch_call)); }

int rch_call_run(const rch_call* call, void* image, void* buffer, const int64_t* jobs, const int64_t* pictures, void* stream) {
    if (int status = check_call(call, image, buffer, jobs)) return status;
    const int64_t base = reinterpret_cast<int64_t>(buffer);
    char* const host = static_cast<char*>(image);
    std::memcpy(host, reinterpret_cast<const void*>(call->template_ptr), static_cast<size_t>(call->image_bytes));

    // Descriptor rows: static fields, buffer offsets made absolute, then this call's addresses.
    int64_t* const rows = reinterpret_cast<int64_t*>(host + call->desc_offset);
    const int64_t* fixed = words(call->rows_ptr);
    const int64_t* relative = words(call->relative_ptr);
    for (int64_t i = 0; i < call->n_rows * kJobColumns; ++i) rows[i] = fixed[i] + relative[i] * base;
    const int64_t extra = call->n_rows - call->n_jobs;
    const int64_t* unpacked = words(call->unpacked_ptr);  // job index of each unpack row
    int64_t picture = 0;
    for (int64_t i = 0; i < call->n_jobs; ++i) {
        const int64_t* in = jobs + i * RCH_CALL_JOB_WORDS;
        int64_t* row = rows + i * kJobColumns;
        bool rows_first = false;  // the job reads the rows that its unpack row writes
        for (int64_t u = 0; u < extra; ++u) {
            if (unpacked[u] != i) continue;
            int64_t* unpack = rows + (call->n_jobs + u) * kJobColumns;
            unpack[RCH_COLUMN(rch_job, src_ptr)] = in[1];
            unpack[RCH_COLUMN(rch_job, dst_ptr)] = row[RCH_COLUMN(rch_job, src_ptr)] = in[10];
            rows_first = true;
        }
        row[RCH_COLUMN(rch_job, dst_ptr)] = in[0];
        if (!rows_first) row[RCH_COLUMN(rch_job, src_ptr)] = in[1];
        if (in[3]) {  // RoPE table: cos, sin and, where the job reads it, the interleaved pairs
            row[RCH_COLUMN(rch_job, cos_ptr)] = in[3];
            row[RCH_COLUMN(rch_job, sin_ptr)] = in[4];
            if (row[RCH_COLUMN(rch_job, pairs_ptr)]) row[RCH_COLUMN(rch_job, pairs_ptr)] = in[5];
        }
        if (in[6]) {  // affine block, in the place its row points to
            std::memcpy(host + (row[RCH_COLUMN(rch_job, scale_ptr)] - base), reinterpret_cast<const void*>(in[6]),
                        static_cast<size_t>(4 * in[7]));
        }
        if (call->prescaled) row[RCH_COLUMN(rch_job, coef_exp)] = in[8];
        if (in[9] > 0) {  // picture offsets from the source base
            const int64_t at = fixed[i * kJobColumns + RCH_COLUMN(rch_job, pic_table_ptr)];
            int64_t table = at;
            for (int64_t u = 0; u < extra; ++u)  // an unpacked job's table belongs to its unpack row
                if (unpacked[u] == i) table = fixed[(call->n_jobs + u) * kJobColumns + RCH_COLUMN(rch_job, pic_table_ptr)];
            int64_t* const out = reinterpret_cast<int64_t*>(host + table);
            for (int64_t p = 0; p < in[9]; ++p) out[p] = pictures[picture + p] - in[1];
            picture += in[9];
        }
    }
    if (call->n_packs > 0) {
        int64_t* const packs = reinterpret_cast<int64_t*>(host + call->packs_offset);
        const int64_t* pack_fixed = words(call->packs_ptr);
        const int64_t* pack_relative = words(call->packs_relative_ptr);
        const int64_t* members = words(call->members_ptr);
        for (int64_t i = 0; i < call->n_packs * kPackColumns; ++i) packs[i] = pack_fixed[i] + pack_relative[i] * base;
        for (int64_t i = 0; i < call->n_packs; ++i)
            packs[i * kPackColumns + RCH_COLUMN(rch_pack, src_ptr)] = jobs[members[i] * RCH_CALL_JOB_WORDS + 2];
    }
    hipStream_t s = as_stream(stream);
    const hipError_t error = hipMemcpyAsync(buffer, image, static_cast<size_t>(call->image_bytes), hipMemcpyHostToDevice, s);
    if (error != hipSuccess) return fail(RCH_E_LAUNCH, "rch_call_run: upload: %s", hipGetErrorString(error));

    const rch_job* table = reinterpret_cast<const rch_job*>(base + call->desc_offset);
    const int n = static_cast<int>(call->n_rows);
    const int32_t* scratch = reinterpret_cast<const int32_t*>(base + call->scratch_offset);
    auto at = [&](int64_t offset) { return reinterpret_cast<const int32_t*>(base + offset); };
    auto i32 = [](int64_t v) { return static_cast<int>(v); };
    for (int64_t l = 0; l < call->n_launches; ++l) {
        const int64_t* L = words(call->launches_ptr) + l * RCH_CALL_LAUNCH_WORDS;
        int status = RCH_OK;
        switch (L[0]) {
            case RCH_CALL_PACK:
                status = rch_basis_pack(reinterpret_cast<const rch_pack*>(base + call->packs_offset), i32(call->n_packs), L[1],
                                        L[2], i32(call->precision), stream);
                break;
            case RCH_CALL_UNPACK:
                status = rch_codes_unpack(table, n, at(L[1]), i32(L[2]), i32(L[3]), stream);
                break;
            case RCH_CALL_DENSE:
                status = rch_rope_store(table, n, at(L[1]), i32(L[2]), i32(L[3]), i32(L[4]), i32(L[5]), stream);
                break;
            case RCH_CALL_RESTORE:
                status = rch_restore(table, n, at(L[1]), i32(L[2]), at(L[3]), i32(L[4]), i32(L[5]), i32(L[6]), i32(L[7]),
                                     i32(L[8]), i32(call->precision), i32(L[9]), i32(L[10]), scratch, stream);
                break;
            case RCH_CALL_PAIR:
                status = rch_restore_pair(table, n, at(L[1]), i32(L[2]), i32(L[3]), at(L[4]), i32(L[5]), i32(L[6]), i32(L[7]),
                                          i32(L[8]), i32(L[9]), i32(call->precision), i32(L[10]), i32(L[11]), scratch, stream);
                break;
            default: status = fail(RCH_E_CONFIG, "rch_call_run: unknown launch kind %lld", static_cast<long long>(L[0]));
        }
        if (status) return status;
    }
    return RCH_OK;
}

}  // extern "C"
