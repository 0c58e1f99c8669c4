// kernels.hpp -- every kernel instantiation the library launches.
//
// The kern_*.hip files instantiate them (one translation unit per family, so
// they compile in parallel); api.hip declares them extern and takes their
// addresses for the launches and occupancy queries.
#pragma once

// bayesr_pipe_kernel<R, layout, fp32, parts>: sequential sweeps over 2-bit codes, slices of up to 1,024 individuals; of
// whole iterations and of parts of one
#define BRR_PIPE_KERNELS_OF(X, F, P)                                                                    \
    X(1, kLayoutDense, F, P) X(1, kLayoutRagged, F, P) X(1, kLayoutEigen, F, P)                         \
    X(2, kLayoutDense, F, P) X(2, kLayoutRagged, F, P) X(2, kLayoutEigen, F, P)

// bayesr_sweep_kernel<R, layout, codes, async, fp32>: the sequential sweeps that the pipelined kernel does not
// take (index lists; four lane runs, whose columns do not fit its LDS ring)
#define BRR_SWEEP_SEQ_KERNELS(X)                                                                        \
    X(1, kLayoutRagged, false, false, false) X(2, kLayoutRagged, false, false, false)                   \
    X(4, kLayoutRagged, false, false, false) X(4, kLayoutDense, true, false, false)                     \
    X(4, kLayoutRagged, true, false, false) X(4, kLayoutEigen, true, false, false)                      \
    X(4, kLayoutDense, true, false, true) X(4, kLayoutRagged, true, false, true)                        \
    X(4, kLayoutEigen, true, false, true)

// asynchronous windows
#define BRR_SWEEP_ASYNC_KERNELS(X)                                                                      \
    X(1, kLayoutDense, true, true, false) X(1, kLayoutRagged, true, true, false)                        \
    X(1, kLayoutRagged, false, true, false) X(1, kLayoutEigen, true, true, false)                       \
    X(2, kLayoutDense, true, true, false) X(2, kLayoutRagged, true, true, false)                        \
    X(2, kLayoutRagged, false, true, false) X(2, kLayoutEigen, true, true, false)                       \
    X(4, kLayoutDense, true, true, false) X(4, kLayoutRagged, true, true, false)                        \
    X(4, kLayoutRagged, false, true, false) X(4, kLayoutEigen, true, true, false)

// bayesr_cohort_kernel<R, fp32, parts>: one or two lane runs per slice (a four-run
// variant gave chains that differ from run to run and stays out)
#define BRR_COHORT_KERNELS(X, P) X(1, false, P) X(2, false, P) X(1, true, P) X(2, true, P)

// bayesr_batch_kernel<NT, dense, fp32>: FP64 residual tiles (up to 16 per slice)
#define BRR_BATCH_KERNELS(X) X(4, true, false) X(4, false, false) X(8, true, false) X(8, false, false) \
    X(13, true, false) X(13, false, false) X(16, true, false) X(16, false, false)
// FP32 residual tiles (up to 32 per slice)
#define BRR_BATCH_F32_KERNELS(X) X(8, true, true) X(8, false, true) X(16, true, true) X(16, false, true) \
    X(25, true, true) X(25, false, true) X(32, true, true) X(32, false, true)

// bayesw_sweep_kernel<R, dense>
#define BRR_BW_KERNELS(X) X(1, true) X(1, false) X(2, true) X(2, false) X(4, true) X(4, false)

#define BRR_SWEEP_INST(R, L, C, A, F) template __global__ void bayesr_sweep_kernel<R, L, C, A, F>(SweepParams);
#define BRR_SWEEP_DECL(R, L, C, A, F) extern template __global__ void bayesr_sweep_kernel<R, L, C, A, F>(SweepParams);
#define BRR_PIPE_INST(R, L, F, P) template __global__ void bayesr_pipe_kernel<R, L, F, P>(SweepParams);
#define BRR_PIPE_DECL(R, L, F, P) extern template __global__ void bayesr_pipe_kernel<R, L, F, P>(SweepParams);
#define BRR_GRAM_INST(M) template __global__ void gram_kernel<M>(GramParams); \
    template __global__ void gram_cohort_kernel<M>(const GramEntry*, uint32_t);
#define BRR_GRAM_DECL(M) extern template __global__ void gram_kernel<M>(GramParams); \
    extern template __global__ void gram_cohort_kernel<M>(const GramEntry*, uint32_t);
#define BRR_COHORT_INST(R, F, P) template __global__ void bayesr_cohort_kernel<R, F, P>(CohortTable);
#define BRR_COHORT_DECL(R, F, P) extern template __global__ void bayesr_cohort_kernel<R, F, P>(CohortTable);
#define BRR_BATCH_INST(NT, D, F) template __global__ void bayesr_batch_kernel<NT, D, F>(BatchParams);
#define BRR_BATCH_DECL(NT, D, F) extern template __global__ void bayesr_batch_kernel<NT, D, F>(BatchParams);
#define BRR_BW_INST(R, D) template __global__ void bayesw_sweep_kernel<R, D>(BwParams);
#define BRR_BW_DECL(R, D) extern template __global__ void bayesw_sweep_kernel<R, D>(BwParams);
