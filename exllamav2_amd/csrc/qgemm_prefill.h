// qgemm_prefill.h -- what the prefill-shaped q_gemm kernels (qgemm_skinny.hip: 17 .. 128 rows, weight-stream bound; qgemm_mfma.hip:
// 256 x 256 tiles, B decoded once per call; qgemm_prefill.hip: the row pre-pass) share with their host driver.
#pragma once
#include "qgemv_common.h"
#include "scratch.h"

struct PrefillArgs
{
    QMatDev m;
    const f16* a;           // [M, K] in packed K order, row stride K (stage_rows_kernel's output)
    f16* c; int ldc;
    const u16* c_invperm;
    int M, c_mode;
};

int stage_rows_plain(const f16* a, int lda, const u16* perm, f16* out, int K, int rows, void* stream);

// qgemm_skinny.hip (17 .. 128 rows): 0 = launched, 1 = does not apply (the many-row kernel takes the call), < 0 = error (message set)
int qgemm_skinny_launch(const PrefillArgs* p, int n, bool gptq, void* stream);     // n <= 3 matrices over the same staged rows

// qgemm_mfma.hip: 0 = launched, < 0 = error (message set)
int qgemm_mfma_launch(const PrefillArgs* p, int n, bool gptq, void* stream);       // n <= 3 matrices over the same staged rows

// four consecutive columns n .. n + 3 of one row of the result: bias, accumulate-into-c, the consumer's column order (JOB: m, c,
// c_invperm, ldc, c_mode)
template <typename JOB> DEV void store_row4(const JOB& job, int row, int n, f32x4 v)
{
    f16* const cp = job.c + (size_t)row * job.ldc;
    if (job.m.bias)
    {
        #pragma unroll
        for (int e = 0; e < 4; e++) v[e] += (float)job.m.bias[n + e];
    }
    if (!job.c_invperm && !(job.ldc & 3) && !(((size_t)job.c) & 7))
    {
        f16x4 h;
        if (job.c_mode == C_ACCUM)
        {
            const f16x4 old = *(const f16x4*)(cp + n);
            #pragma unroll
            for (int e = 0; e < 4; e++) v[e] += (float)old[e];
        }
        #pragma unroll
        for (int e = 0; e < 4; e++) h[e] = (f16)v[e];
        *(f16x4*)(cp + n) = h;
        return;
    }
    #pragma unroll
    for (int e = 0; e < 4; e++)
    {
        const int nn = job.c_invperm ? (int)job.c_invperm[n + e] : n + e;
        float w = v[e];
        if (job.c_mode == C_ACCUM) w += (float)cp[nn];
        cp[nn] = (f16)w;
    }
}
