// instances.hpp -- the transform kernels of one compiled length L as explicit instantiations:
// defined by instances.hip, compiled once per length so that the lengths build in parallel,
// declared (EXT = extern) for the library's own translation unit.
#pragma once
#include "k_cheb_dmfma.hpp"
#include "k_cheb_mfma.hpp"
#include "k_transform.hpp"

// span transforms, precision R (all that RPCF_SPAN_ONLY_LENGTH has)
#define RPCF_INSTANCES_SPAN(EXT, L, R)                                                                                \
    EXT template __global__ void k_span_inv<L, R>(const cplx<R>*, long, long, cplx<R>*, long, long, Dims, int, FftPlan, \
                                                  int, int, const int*);                                               \
    EXT template __global__ void k_span_fwd<L, R>(const cplx<R>*, long, long, int, cplx<R>*, long, long, Dims, int,     \
                                                  FftPlan, int, int, const int*, int*);
// x and span transforms (all that an RPCF_XY_LENGTHS length has, in FP64)
#define RPCF_INSTANCES_XY(EXT, L, R)                                                                                  \
    RPCF_INSTANCES_SPAN(EXT, L, R)                                                                                     \
    EXT template __global__ void k_lamb_phys<L, R>(const cplx<R>*, long, long, cplx<R>*, long, long, int, const double*, \
                                                   long, double, Dims, FftPlan, int, int, Members);
// Chebyshev transforms of length 2N = L with the padded side in precision R
#define RPCF_INSTANCES_CHEB(EXT, L, R)                                                                                 \
    EXT template __global__ void k_cheb_s2p<1, L, R>(const double2*, long, long, cplx<R>*, long, long, Dims, FftPlan,  \
                                                     const double2*, int, int, const int*);                            \
    EXT template __global__ void k_cheb_s2p_h<(L >= 64 ? L : 64), R>(const double2*, long, long, cplx<R>*, long, long, \
                                                                     Dims, const double2*, int, const int*);           \
    EXT template __global__ void k_p2s_nl2<L, R>(const cplx<R>*, long, long, double2*, long, Dims, FftPlan,            \
                                                 const double2*, int, int, Members);                                   \
    EXT template __global__ void k_p2s_nl<L, R>(const cplx<R>*, long, long, double2*, long, Dims, FftPlan,             \
                                                const double2*, int, int, Members);
#define RPCF_INSTANCES(EXT, L)                                                                                         \
    RPCF_INSTANCES_XY(EXT, L, double)                                                                                  \
    RPCF_INSTANCES_XY(EXT, L, float)                                                                                   \
    RPCF_INSTANCES_CHEB(EXT, L, double)                                                                                \
    RPCF_INSTANCES_CHEB(EXT, L, float)                                                                                 \
    EXT template __global__ void k_cheb_s2p<0, L, double>(const double2*, long, long, double2*, long, long, Dims,      \
                                                          FftPlan, const double2*, int, int, const int*);              \
    EXT template __global__ void k_x_c2r<L>(const double2*, double*, Dims, FftPlan, int, int);                         \
    EXT template __global__ void k_velocity_tile<L, double2>(const double2*, const double2*, long, double2*, long,     \
                                                             long, Dims, Members, int, int);                           \
    EXT template __global__ void k_velocity_tile<L, float2>(const double2*, const double2*, long, float2*, long, long, \
                                                            Dims, Members, int, int);                                  \
    EXT template __global__ void k_s2p_mfma<L>(const float2*, long, long, float2*, long, long, Dims, \
                                                                  const h8_t*, const int*, int);                       \
    EXT template __global__ void k_p2s_mfma<L>(const float2*, long, long, double2*, long, Dims,     \
                                                                  const h8_t*, int, int, Members);                     \
    EXT template __global__ void k_p2s_dmfma<L, cheb_dmfma::kChunk>(const double2*, long, long, double2*, long, Dims, \
                                                                          const double*, Members, int, int); \
    EXT template __global__ void k_p2s_dmfma<L, cheb_dmfma::kChunkMany>(const double2*, long, long, double2*, long, Dims, \
                                                                          const double*, Members, int, int);
