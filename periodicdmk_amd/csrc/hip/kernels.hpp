// gfx950 kernels of the periodic DMK evaluate() path.  Included by plan.hip only.
//
// Stage map (reference functions each kernel replaces):
//   k_gather_charges ... update_charges + image-charge gather
//                        (cpp/src/periodic_dmk.cpp:164-170, cpp/src/dmk/pbc_tree.cpp:1807-1821)
//   k_charge2proxy ..... proxy::charge2proxycharge_3d (cpp/src/dmk/proxy.cpp:153-212)
//   k_tensor3 .......... tensorprod::transform_3d c2p / p2c (cpp/src/dmk/tensorprod.cpp:39-75)
//   k_proxy2pw ......... proxy::proxycharge2pw_3d (cpp/src/dmk/proxy.cpp:42-90)
//   k_pw_shift ......... form_eval_expansions shifts with fused radialft
//                        (cpp/src/dmk/pbc_tree.cpp:1294-1369, cpp/include/dmk/tree.hpp:287-316)
//   k_pw2proxy ......... planewave_to_proxy_potential (cpp/src/dmk/planewave.cpp:49-105)
//   k_eval_targets ..... proxy::eval_targets_3d (cpp/src/dmk/proxy.cpp:307-448)
//   k_near_field ....... evaluate_direct_interactions + laplace_3d_poly_all_pairs
//                        (cpp/src/dmk/pbc_tree.cpp:1442-1681, cpp/include/dmk/vector_kernels.hpp:354-421)
//   k_ff_* ............. far_field_nufft, 3-D non-QP (cpp/src/dmk/pbc.cpp:378-541)
//   k_finalize ......... apply_target_self_correction + desort_potentials + far-field add
//                        (cpp/src/dmk/pbc_tree.cpp:1759-1805, cpp/src/periodic_dmk.cpp:172-182)
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>
#include <utility>

#include "dpp_fma.hpp"

namespace pdmk::gpu {

template <class R>
struct alignas(4 * sizeof(R)) P4 { R x, y, z, w; };

template <class R>
struct alignas(2 * sizeof(R)) Cx { R re, im; };

// Workgroups are dispatched to the 8 XCDs round-robin; this bijection of [0, nb) gives each
// XCD one contiguous range of workgroup indices, so work items that share inputs (items are
// laid out in tree order, i.e. spatially) run under the same L2.
__device__ __forceinline__ int xcd_block(int b, int nb) {
    constexpr int X = 8;
    const int x = b % X, i = b / X, q = nb / X, r = nb % X;
    return x * q + min(x, r) + i;
}

// Kernels of the proxy / plane-wave chain raise their waves' issue priority: evaluate()
// runs them beside the near-field kernel, and the chain is the longer path.
__device__ __forceinline__ void chain_priority() { __builtin_amdgcn_s_setprio(2); }

// A zero the compiler cannot see through: adding it moves a wave-uniform value into a VGPR.
__device__ __forceinline__ int vgpr_zero() {
    int z;
    asm volatile("v_mov_b32 %0, 0" : "=v"(z));
    return z;
}

// 1 / sqrt(x) for the near-field distances: every caller passes 1e-30 < x < 1e30 (a positive
// normal number).  FP64: the hardware estimate y = v_rsq_f64(x) and one third-order
// correction y (1 + e/2 + 3e^2/8), e = 1 - x y^2 -- the library rsqrt's own arithmetic, bit
// for bit on this range, without its branches for zero, infinity and NaN inputs.
template <class R> __device__ __forceinline__ R rsqrt_full(R x);
template <> __device__ __forceinline__ float rsqrt_full<float>(float x) { return __frsqrt_rn(x); }
template <> __device__ __forceinline__ double rsqrt_full<double>(double x) {
    const double y = __builtin_amdgcn_rsq(x);
    const double e = fma(y * -x, y, 1.0);
    return fma(y * e, fma(e, 0.375, 0.5), y);
}

// ------------------------------------------------------------------ O(N) stages
// Charges of the sorted sources.
template <class R>
__global__ void k_gather_charges(const double *__restrict__ q, const int *__restrict__ src_user, P4<R> *__restrict__ src,
                                 int nsall, R *__restrict__ pot_sorted, R *__restrict__ pot_near, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < nsall) src[i].w = (R)q[src_user[i]];
    if (i < n) {
        pot_sorted[i] = R(0);
        pot_near[i] = R(0);
    }
}

// Quasi-periodic trees: the charges times the real and the imaginary part of their image phase
// e^{i b.R} (originals: phase 1), each in a copy of the sources (ld apart), and both
// components' potentials cleared.
template <class R>
__global__ void k_gather_qp(const double *__restrict__ q, const int *__restrict__ src_user,
                            const double2 *__restrict__ phase, P4<R> *__restrict__ src, long long ld, int nsall,
                            R *__restrict__ pot_sorted, R *__restrict__ pot_near, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < nsall) {
        const double v = q[src_user[i]];
        const double2 ph = phase[i];
        src[i].w = (R)(v * ph.x);
        src[ld + i].w = (R)(v * ph.y);
    }
    if (i < 2 * n) {
        pot_sorted[i] = R(0);
        pot_near[i] = R(0);
    }
}

// out[2 u], out[2 u + 1] = Re, Im: the two components' chain and near-field potentials, the self
// correction on the real one (the originals' charges are real), rounded to R, and the complex
// far field added to that.
template <class R>
__global__ void k_finalize_qp(const R *__restrict__ pot_sorted, const R *__restrict__ pot_near, const double *__restrict__ w0,
                              const int *__restrict__ trg_user, const double *__restrict__ q,
                              const double2 *__restrict__ far, R *__restrict__ out, int n, int use_self, int use_far) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int u = trg_user[i];
    double re = (double)pot_sorted[i] + (double)pot_near[i], im = (double)pot_sorted[n + i] + (double)pot_near[n + i];
    if (use_self) re -= w0[i] * q[u];
    double2 f = make_double2(0, 0);
    if (use_far) f = far[u];
    out[2 * (size_t)u] = (R)((double)(R)re + f.x);
    out[2 * (size_t)u + 1] = (R)((double)(R)im + f.y);
}

// pot[u] = pot_sorted[i] - w0_i q_u + far[u], u = trg_user[i].  Vector v = blockIdx.z of a many-vector launch uses the
// arrays offset by v times the vs_* element strides (all zero for one vector).
template <class R>
__global__ void k_finalize(const R *__restrict__ pot_sorted, const R *__restrict__ pot_near, const double *__restrict__ w0,
                           const int *__restrict__ trg_user, const double *__restrict__ q, const double *__restrict__ far,
                           const int *__restrict__ far_idx, R *__restrict__ pot, int n, int use_self, int use_far,
                           long long vs_sorted = 0, long long vs_near = 0, long long vs_q = 0,
                           long long vs_far = 0, long long vs_pot = 0) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const long long vz = blockIdx.z;
    pot_sorted += vz * vs_sorted;
    pot_near += vz * vs_near;
    q += vz * vs_q;
    far += vz * vs_far;
    pot += vz * vs_pot;
    const int u = trg_user[i];
    double v = (double)pot_sorted[i] + (double)pot_near[i];
    if (use_self) v -= w0[i] * q[u];
    if (use_far) v += far[far_idx[i]];
    pot[u] = (R)v;
}

typedef double c2p_d4 __attribute__((ext_vector_type(4)));
typedef float c2p_f4 __attribute__((ext_vector_type(4)));

// 16 x 16 x 4 matrix-core products.  Operands: lane l holds A[l%16][l/16] and B[l/16][l%16].
// Accumulator element e of lane l is D[row(l/16, e)][l%16]: rows l/16 + 4e for FP64 and
// 4(l/16) + e for FP32 (both read off the hardware with in-bounds probes).
template <class R> struct Mfma16;
template <> struct Mfma16<double> {
    typedef c2p_d4 acc_t;
    static __device__ __forceinline__ acc_t mma(double a, double b, acc_t c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int kk, int e) { return kk + 4 * e; }
};
template <> struct Mfma16<float> {
    typedef c2p_f4 acc_t;
    static __device__ __forceinline__ acc_t mma(float a, float b, acc_t c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int kk, int e) { return 4 * kk + e; }
};
// ------------------------------------------------------------------ upward pass
// One destination box per workgroup (or per `parts` workgroups):
//   C[c][b][a] = sum_s T_a(x_s) T_b(y_s) T_c(z_s) q_s,  x_s = sc (r_s - centre).
// Sources hold coordinates relative to their leaf centre; each range lies in one leaf and
// carries rng_off = leaf centre - box centre, so x_s = sc (local_s + off).
//
// Per box this is a GEMM of P^2 columns (c, b) by P values of a over the sources, on the matrix
// cores with 4-wide blocks, which pad a to a multiple of 4 (18 to 20, 28 and 28): the 16-wide
// products used before at p = 28 pad it to 32, and at p = 18 that waste kept both precisions on
// the vector ALUs, in competition with the near field.  Each output is the chain of fused
// multiply-adds over the sources in order, as on the vector ALUs, bit for bit (checked on
// gfx950: v_mfma_f32_4x4x1 adds one product per step, v_mfma_f64_4x4x4 four in k order).
//   FP32, v_mfma_f32_4x4x1 (16 blocks): lane l owns column 64 w + l; its factor q T_b T_c of
//     a source is the B operand, and T_a comes as an A operand that broadcasts one block of 4
//     lanes to all (cbsz 4), so one register with the T_a of SPA sources serves SPA G products.
//   FP64, v_mfma_f64_4x4x4 (4 blocks): a tile of 16 columns by 4 values of a over 4 sources;
//     lane (k, blk, i) = (l / 16, l / 4 % 4, l % 4) supplies A = q T_b T_c of column 4 blk + i and
//     B = T_(4 g + i), both at source k, and holds D[column 4 blk + l / 16][a = 4 g + i].
// Box g's sources are items grp_ptr[g] .. (source, range), its ranges without a break (short leaves
// fill a tile together, and a tile's loads wait for no walk over the ranges); their Chebyshev values are tabulated in LDS, two buffers in turn: the next tile's
// points load while the current one's products run.
//
// Alone, N = 1e6 (576 boxes): FP32 6 digits 305 -> 223 us, FP64 475 -> 355, 9 digits 975 -> 887
// (evaluate() 6959 -> 6600); N = 3e4 (64 boxes) 72 -> 34,
// 81 -> 29, 137 -> 69; clustered, 9 digits N = 1e6 7675 -> 7387, 12 digits N = 1.5e5 2246 -> 1118.
// Bound by the matrix cores and, with 576 boxes for 256 CUs, by the last round of boxes.
template <class R, int P> struct C2pCfg {
    static constexpr bool F32 = sizeof(R) == 4;
    static constexpr int G = (P + 3) / 4, PX = 4 * G;     // groups of 4 values of a
    static constexpr int CB = P * P;                      // columns (c, b)
    static constexpr int CW = F32 ? 64 : 16;              // columns of a tile
    static constexpr int CT = (CB + CW - 1) / CW;         // column tiles
    // waves per workgroup.  FP64 at p = 28, 38: 4, one per SIMD, and two workgroups or more per CU
    // (7 waves of 7 tiles: N = 1e6 9 digits 1012 us, clustered 8942; 5 waves: 1304).  FP64 at p = 9: 3
    // waves of 2 tiles, which find room beside the near field; workgroups of 7 waited for it (N = 2e5,
    // 3888 boxes: evaluate() 571 -> 481 us; 1.5e5, 576 boxes 338 -> 306)
    static constexpr int NW = F32 ? (CT > 16 ? (CT + 1) / 2 : CT) : (P == 9 ? 3 : (P == 18 ? 7 : 4));
    static constexpr int parts(int tpw) { return (CT + NW * tpw - 1) / (NW * tpw); }  // workgroups per box
    static constexpr int SPA = F32 ? 64 / PX : 4;         // sources per A register / product
    static constexpr int TS = F32 ? 60 / SPA * SPA : 32;  // sources per table
    // LDS rows: x values, then y and z (odd, so that the rows of a fragment spread over the banks)
    static constexpr int SX = F32 ? PX : PX + 1, SY = P | 1;
    static constexpr int buf = TS * (SX + 2 * SY);        // elements of a buffer
    static constexpr int NTK = (3 * TS + 64 * NW - 1) / (64 * NW);  // table tasks per thread
};

// items of the ranges: item[rng_ptr[r] + i] = (rng_begin[r] + i, r), a wavefront per range
__global__ __launch_bounds__(256) void k_c2p_items(const int *__restrict__ rng_begin, const int *__restrict__ rng_count,
                                                   const int *__restrict__ rng_ptr, int n_rng, int2 *__restrict__ item) {
    const int r = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (r >= n_rng) return;
    const int beg = rng_begin[r], cnt = rng_count[r], o = rng_ptr[r];
    for (int i = threadIdx.x & 63; i < cnt; i += 64) item[o + i] = make_int2(beg + i, r);
}

// SPA G products of one A register, its blocks in turn: sources s, values 4 g .. 4 g + 3
template <int G, int... I>
__device__ __forceinline__ void c2p_products(float a, const float *w, c2p_f4 *acc, std::integer_sequence<int, I...>) {
    ((acc[I % G] = __builtin_amdgcn_mfma_f32_4x4x1f32(a, w[I / G], acc[I % G], 4, I, 0)), ...);
}

// TPW: column tiles per wave (FP32: 1); tile (part NW + w) + parts NW m of wave w
template <class R, int P, int TPW>
__global__ __launch_bounds__((64 * C2pCfg<R, P>::NW), 2) void k_charge2proxy(
    const P4<R> *__restrict__ src, const int *__restrict__ grp_slot, const R *__restrict__ grp_geom,
    const int *__restrict__ grp_ptr, const int2 *__restrict__ item, const R *__restrict__ rng_off,
    R *__restrict__ proxy, const R *__restrict__ qv = nullptr, int qv_ld = 0,
    long long vs_out = 0, long long vs_src = 0) {
    chain_priority();
    using C = C2pCfg<R, P>;
    constexpr int G = C::G, NW = C::NW, TS = C::TS, SX = C::SX, SY = C::SY, SPA = C::SPA, NTK = C::NTK, CB = C::CB;
    constexpr int parts = C::parts(TPW);
    constexpr bool F32 = C::F32;
    static_assert(!F32 || TPW == 1, "one column per lane");
    // vector blockIdx.z of a launch for several: its sources at src + z vs_src, or its charges at
    // qv[source * qv_ld + z] (src[].w otherwise); its proxies vs_out elements further on
    src += (long long)blockIdx.z * vs_src;
    proxy += (long long)blockIdx.z * vs_out;
    __shared__ R lds[2 * C::buf];
    const int g = blockIdx.x / parts, part = blockIdx.x - g * parts, lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const R sc = grp_geom[4 * g + 3];
    // this lane's columns: table offsets of b and c (columns past the last repeat column 0)
    int ob[TPW], oc[TPW];
#pragma unroll
    for (int m = 0; m < TPW; ++m) {
        const int col = ((part * NW + w) + parts * NW * m) * C::CW + (F32 ? lane : (lane & 15));
        ob[m] = col < CB ? col % P : 0;
        oc[m] = col < CB ? col / P : 0;
    }
    static_assert(F32 || C::CT > (TPW - 1) * NW * parts, "every wave has its first TPW - 1 tiles");
    const int nt = (C::CT - (part * NW + w) + parts * NW - 1) / (parts * NW);  // this wave's tiles
    c2p_f4 accf[F32 ? G : 1];
    double accd[F32 ? 1 : TPW][F32 ? 1 : G];
    if constexpr (F32) {
#pragma unroll
        for (int i = 0; i < G; ++i) accf[i] = c2p_f4{0, 0, 0, 0};
    } else {
#pragma unroll
        for (int m = 0; m < TPW; ++m)
#pragma unroll
            for (int i = 0; i < G; ++i) accd[m][i] = 0;
    }
    const int i1 = grp_ptr[g + 1];
    int i0 = grp_ptr[g];  // the next tile's first source
    R px[NTK], pq[NTK];
    // next tile's points into registers (task t: component t / TS of source t % TS; past the end:
    // charge 0)
    auto fetch = [&]() {
#pragma unroll
        for (int i = 0; i < NTK; ++i) {
            const int t = (int)threadIdx.x + 64 * NW * i, s = t % TS, d = t / TS;
            px[i] = R(0);
            pq[i] = R(0);
            if (i0 + s < i1 && d < 3) {
                const int2 e = item[i0 + s];
                const R *x = reinterpret_cast<const R *>(src + e.x);
                px[i] = x[d] + rng_off[4 * e.y + d];
                pq[i] = d == 2 ? (qv ? qv[(size_t)e.x * qv_ld + blockIdx.z] : x[3]) : R(1);
            }
        }
    };
    auto tabulate = [&](R *T0) {
#pragma unroll
        for (int i = 0; i < NTK; ++i) {
            const int t = (int)threadIdx.x + 64 * NW * i, s = t % TS, d = t / TS;
            if (d >= 3) break;
            R *T = d == 0 ? T0 + s * SX : T0 + TS * SX + ((d - 1) * TS + s) * SY;
            const R x = sc * px[i], m = pq[i];
            R t0 = m, t1 = x * m;
            T[0] = t0;
            T[1] = t1;
#pragma unroll
            for (int k = 2; k < P; ++k) {
                const R t2 = R(2) * x * t1 - t0;
                T[k] = t2;
                t0 = t1;
                t1 = t2;
            }
            if (d == 0)
                for (int k = P; k < C::PX; ++k) T[k] = R(0);
        }
    };
    fetch();
    for (int it = 0; i0 < i1; ++it) {
        R *T0 = lds + (it & 1) * C::buf;
        tabulate(T0);
        const int cur = min(TS, i1 - i0);
        i0 += TS;
        fetch();
        // (one barrier per tile: a wave that is a tile ahead writes the other buffer, and a buffer is
        // written again only after the barrier that follows its last reads)
        __syncthreads();
        const R *Tx = T0, *Ty = T0 + TS * SX, *Tz = Ty + TS * SY;
        if constexpr (F32) {
            for (int s0 = 0; s0 < cur; s0 += SPA) {
                const float a = Tx[s0 * SX + lane];  // (lanes past SPA rows: in no product's block)
                float wv[SPA];
#pragma unroll
                for (int i = 0; i < SPA; ++i) wv[i] = Ty[(s0 + i) * SY + ob[0]] * Tz[(s0 + i) * SY + oc[0]];
                c2p_products<G>(a, wv, accf, std::make_integer_sequence<int, SPA * G>{});
            }
        } else {
            const int kk = lane >> 4, j = lane & 3;
            for (int s0 = 0; s0 < cur; s0 += 4) {
                const int s = s0 + kk;
                double b[G];
#pragma unroll
                for (int i = 0; i < G; ++i) b[i] = Tx[s * SX + 4 * i + j];
#pragma unroll
                for (int m = 0; m < TPW; ++m) {
                    // (only the last tile of some waves may be past the end; wave-uniform)
                    if (C::CT % (NW * parts) != 0 && m == TPW - 1 && m >= nt) break;
                    const double a = Ty[s * SY + ob[m]] * Tz[s * SY + oc[m]];
#pragma unroll
                    for (int i = 0; i < G; ++i) accd[m][i] = __builtin_amdgcn_mfma_f64_4x4x4f64(a, b[i], accd[m][i], 0, 0, 0);
                }
            }
        }
    }
    R *out = proxy + (size_t)grp_slot[g] * (P * P * P);
    if constexpr (F32) {
        const int col = (part * NW + w) * 64 + lane;
        if (col < CB) {
#pragma unroll
            for (int a = 0; a < P; ++a) out[(size_t)col * P + a] = accf[a >> 2][a & 3];
        }
    } else {
#pragma unroll
        for (int m = 0; m < TPW; ++m) {
            const int col = ((part * NW + w) + parts * NW * m) * 16 + (lane & 12) + (lane >> 4);
#pragma unroll
            for (int i = 0; i < G; ++i) {
                const int a = 4 * i + (lane & 3);
                if (col < CB && a < P) out[(size_t)col * P + a] = accd[m][i];
            }
        }
    }
}

// ------------------------------------------------------------------ tensor transforms
// All transforms are sequences of mode products of a small 3-D tensor with small dense
// matrices.  One workgroup owns one output box; a thread owns one column of the mode being
// contracted (the column sits in registers), the matrix entries are read with wave-uniform
// addresses (scalar loads), and intermediates live in LDS with row strides of an odd number
// of elements, so 64-bit LDS accesses by consecutive lanes hit distinct banks.  When the
// intermediates of a whole box do not fit the LDS budget the box is processed in slices of
// the first contraction's output index (upward, c2p/p2c) or of the first output index of the
// downward contraction; each slice then runs all three steps on its own.
constexpr int kTfLdsBytes = 64 * 1024;

template <int N> struct OddStride { static constexpr int v = (N % 2) ? N : N + 1; };

// LDS budget of a tensor-transform workgroup: 64 KiB, or all 160 KiB of a CU for FP64 at
// p >= 38 (12 digits), whose registers allow one such workgroup per CU anyway: 6 output planes
// per workgroup instead of 1, so each input is read 7 times instead of 38 (measured on the
// N=4e6 clustered workload: child -> parent 431 -> 128 ms, parent -> child 162 -> 73 ms per
// evaluate).  The proxy <-> plane-wave transforms keep 64 KiB: with 160 KiB they hold one
// wavefront per SIMD and ran 1.7x slower.
constexpr int tf_lds_budget(int p, int real_bytes) { return p >= 38 && real_bytes == 8 ? 160 * 1024 : kTfLdsBytes; }

// slices per pass so that `reserved` + `per_slice` bytes x slices stays within the LDS budget
constexpr int tf_slices(int total, int per_slice, int reserved = 0, int budget = kTfLdsBytes) {
    const int k = (budget - reserved) / per_slice;
    return k < 1 ? 1 : (k > total ? total : k);
}

// Slices of the proxy <-> plane-wave transforms that fit the LDS budget; each slice is a
// workgroup of its own (grid y), so a level with few boxes still fills the GPU.
// BK: the LDS budget in KiB per workgroup (0 = the default below); the autotuner picks
// among 0, 16, 32 and 64 per plan.
// slices per box from which the proxy <-> plane-wave transforms take their first contraction
// of whole boxes from HBM (two passes) rather than re-reading each box's input per slice
constexpr int kTwoPassSlices = 8;

template <class R, int P, int NPW, int BK = 0> struct P2pwCfg {
    static constexpr int H = (NPW + 1) / 2;
    // (FP64 at p = 28: one k3 plane per workgroup, 31 KB, five workgroups per CU; two planes at
    // 61 KB fit two: N=1e6 9-digit evaluate() 9.06 -> 8.95 ms.  At p = 18 a 32 KB budget, on
    // the plane-wave -> proxy side too: FP32 4 planes instead of 9, 6-digit evaluate()
    // 3.06 -> 2.95 ms; FP64 2 instead of 4, 4.72 -> 4.60 ms)
    static constexpr int K3 = tf_slices(H, (P * P + NPW * OddStride<P>::v) * (int)sizeof(Cx<R>), 0,
                                        BK ? BK * 1024 : (((P == 28 && sizeof(R) == 8) || P == 18) ? 32 * 1024 : kTfLdsBytes));
    static constexpr int slices = (H + K3 - 1) / K3;
    // the y and x steps have K3 P and K3 n columns of n outputs for 256 threads; the outputs
    // of a column are split over SGY / SGX wavefronts when that fills more of them
    static constexpr int NT = 256;
    static constexpr int cap(int v) { return v < 1 ? 1 : (v > 8 ? 8 : v); }
    static constexpr int SGY = cap(NT / ((K3 * P + 63) / 64 * 64)), SGX = cap(NT / ((K3 * NPW + 63) / 64 * 64));
    static constexpr int PSY = (NPW + SGY - 1) / SGY, PSX = (NPW + SGX - 1) / SGX;
};
template <class R, int P, int NPW, int BK = 0> struct Pw2pCfg {
    static constexpr int H = (NPW + 1) / 2;
    // (FP64 at p = 28: 2 slices of a per workgroup, 43 KB, so three workgroups share a CU;
    // 3 per workgroup at 65 KB fit two: N=1e6 9-digit evaluate() 9.12 -> 9.07 ms.  p = 18: 32 KB in
    // FP64, 16 KB in FP32 (3 slices): the FP32 chain alone 81 -> 67 us at N = 1e3, 175 -> 152 at 3e4,
    // 638 -> 576 at 2.5e5; FP64 at 16 KB 75 -> 84 and 817 -> 896)
    static constexpr int AC = tf_slices(P, (H * NPW + H * OddStride<P>::v) * (int)sizeof(Cx<R>), 0,
                                        BK ? BK * 1024 : ((P == 28 && sizeof(R) == 8) ? 48 * 1024 : (P == 18 ? (int)sizeof(R) * 4096 : kTfLdsBytes)));
    static constexpr int slices = (P + AC - 1) / AC;
    // the y and z steps have AC H and AC P columns of P outputs for 256 threads; the outputs of
    // a column are split over SGY / SGZ wavefronts when that fills more of them
    static constexpr int NT = 256;
    static constexpr int cap(int v) { return v < 1 ? 1 : (v > 8 ? 8 : v); }
    static constexpr int SGY = cap(NT / ((AC * H + 63) / 64 * 64)), SGZ = cap(NT / ((AC * P + 63) / 64 * 64));
    static constexpr int PSY = (P + SGY - 1) / SGY, PSZ = (P + SGZ - 1) / SGZ;
};

// 3-mode tensor transform out(a',b',c') (+)= sum_children U0(a',a) U1(b',b) U2(c',c) in(a,b,c)
// (tensor layout [c][b][a], a fastest).  U_d is the minus/plus parent<->child matrix selected
// by bit d of the child code, transposed for child -> parent.  Item i writes out slot
// item_out[i] from the CSR range item_ptr[i]..item_ptr[i+1] of (in slot, child code);
// item_add[i] = accumulate into the existing output.  Workgroup (item, slice) computes the
// output planes c' in [slice kc, slice kc + kc), kc <= T3Cfg::KC; the grid is 1-D, workgroup
// (item, slice) at xcd_block index item * slices + slice, so an item's slices run together
// under one L2 and its input is fetched from memory about once.
template <class R, int P> struct T3Cfg {
    static constexpr int PP = P * P, TS = OddStride<P>::v;
    // output planes per workgroup (the budget keeps 2 p^2 values spare, so FP64 at p = 28
    // fits three workgroups per CU)
    static constexpr int KC = tf_slices(P, (PP + P * TS) * (int)sizeof(R), 2 * PP * (int)sizeof(R),
                                        tf_lds_budget(P, (int)sizeof(R)));
    // at most 4 waves below p = 38: evaluate() runs these beside the near field, whose
    // retiring 4-wave workgroups free 4 wave slots at a time
    static constexpr int threads = PP <= 256 ? (PP + 63) / 64 * 64 : (P >= 38 ? 512 : 256);
    // the y and x steps have KC P columns of P outputs; when that leaves more than half the
    // threads idle, each column's outputs are split between SG wavefronts
    static constexpr int SG = KC * P * 2 <= threads ? 2 : 1;
    static constexpr int PS = (P + SG - 1) / SG;  // outputs per thread in the y and x steps
    static constexpr int slots(int nk) { return (nk * P + 63) / 64 * 64 * SG; }  // y / x work slots
};

// Work slot w of the y and x steps -> (column, segment): consecutive lanes take consecutive
// columns, and a wavefront's lanes share one segment (so its matrix rows are wave-uniform).
template <int SG> __device__ __forceinline__ void t3_slot(int w, int &col, int &sg) {
    col = (w & 63) + 64 * (w / (64 * SG));
    sg = __builtin_amdgcn_readfirstlane((w >> 6) % SG);  // wave-uniform (w = lane + multiple of 64)
}

template <class R, int P, bool TRANSPOSE>
__global__ __launch_bounds__((T3Cfg<R, P>::threads)) void k_tensor3(
    const R *__restrict__ in_base, R *__restrict__ out_base, const int *__restrict__ item_out,
    const int *__restrict__ item_add, const int *__restrict__ item_ptr, const int *__restrict__ in_slot,
    const int *__restrict__ in_code, const R *__restrict__ mats_rm, int n_items, int kc, long long vs_in = 0,
    long long vs_out = 0) {
    chain_priority();
    in_base += (long long)blockIdx.z * vs_in;  // vector blockIdx.z of a many-vector launch
    out_base += (long long)blockIdx.z * vs_out;
    using Cfg = T3Cfg<R, P>;
    constexpr int PP = P * P, TS = Cfg::TS, KC = Cfg::KC, NT = Cfg::threads, SG = Cfg::SG, PS = Cfg::PS;
    constexpr int PR = P;  // row stride of the matrices
    constexpr int XC = (Cfg::slots(KC) + NT - 1) / NT;
    __shared__ R T1[KC * PP];       // [k][b][a]
    __shared__ R T2[KC * P * TS];   // [k][b'][a] rows of TS
    // U_s(r, c) = M_s[r + P c] (parent -> child) or M_s[c + P r] (child -> parent), read
    // row-major from mats_rm[(transposed) 2 + s][r][c] at wave-uniform addresses: scalar
    // loads into SGPRs (a broadcast LDS read of 16 bytes would feed only 2 FP64 / 4 FP32 FMAs
    // per lane)
    const int ns = (P + kc - 1) / kc, lg = xcd_block(blockIdx.x, gridDim.x);
    const int it = lg / ns;
    if (it >= n_items) return;
    const int k0 = (lg - it * ns) * kc;
    const R *Ubase = mats_rm + (TRANSPOSE ? 2 : 0) * PP;
    const int nk = min(kc, P - k0), nslot = Cfg::slots(nk);
    R *out = out_base + (size_t)item_out[it] * P * PP;
    const bool add = item_add[it] != 0;
    const int e0 = item_ptr[it], e1 = item_ptr[it + 1];
    // s += sum_c U(r, c) x[c] for the row of U starting at urow
    auto row_dot = [](const R *urow, const R (&x)[P], R s) {
#pragma unroll
        for (int c = 0; c < P; ++c) s = fma(urow[c], x[c], s);
        return s;
    };
    // the same sums for four consecutive rows at once (four independent dependency chains)
    auto row_dot4 = [](const R *urow, const R (&x)[P], R (&o)[4]) {
#pragma unroll
        for (int i = 0; i < 4; ++i) o[i] = R(0);
#pragma unroll
        for (int c = 0; c < P; ++c)
#pragma unroll
            for (int i = 0; i < 4; ++i) o[i] = fma(urow[i * PR + c], x[c], o[i]);
    };
    // x-step accumulators: work slot (column (k, b'), segment of a') -- persistent over children
    R acc[XC][PS];
#pragma unroll
    for (int q = 0; q < XC; ++q)
#pragma unroll
        for (int a = 0; a < PS; ++a) acc[q][a] = R(0);
    for (int e = e0; e < e1; ++e) {
        const R *in = in_base + (size_t)in_slot[e] * P * PP;
        const int code = in_code[e];
        const R *U0 = Ubase + (code & 1) * P * PR, *U1 = Ubase + ((code >> 1) & 1) * P * PR,
                *U2 = Ubase + ((code >> 2) & 1) * P * PR;
        __syncthreads();
        // z: T1[k][b][a] = sum_c U2(k0 + k, c) in[c][b][a]
        for (int j = threadIdx.x; j < PP; j += NT) {
            R x[P];
#pragma unroll
            for (int c = 0; c < P; ++c) x[c] = in[c * PP + j];
            int k = 0;
            for (; k + 4 <= nk; k += 4) {  // four independent sums at a time
                R o[4];
                row_dot4(U2 + (k0 + k) * PR, x, o);
#pragma unroll
                for (int i = 0; i < 4; ++i) T1[(k + i) * PP + j] = o[i];
            }
            for (; k < nk; ++k) T1[k * PP + j] = row_dot(U2 + (k0 + k) * PR, x, R(0));
        }
        __syncthreads();
        // y: T2[k][b'][a] = sum_b U1(b', b) T1[k][b][a]; slot = (column (k, a), segment of b')
        for (int w = threadIdx.x; w < nslot; w += NT) {
            int col, sg;
            t3_slot<SG>(w, col, sg);
            if (col >= nk * P) continue;
            const int k = col / P, a = col - k * P;
            R x[P];
#pragma unroll
            for (int b = 0; b < P; ++b) x[b] = T1[k * PP + b * P + a];
            const int b2e = min(P, sg * PS + PS);
            int b2 = sg * PS;
            for (; b2 + 4 <= b2e; b2 += 4) {
                R o[4];
                row_dot4(U1 + b2 * PR, x, o);
#pragma unroll
                for (int i = 0; i < 4; ++i) T2[(k * P + b2 + i) * TS + a] = o[i];
            }
            for (; b2 < b2e; ++b2) T2[(k * P + b2) * TS + a] = row_dot(U1 + b2 * PR, x, R(0));
        }
        __syncthreads();
        // x: acc[a'] += sum_a U0(a', a) T2[k][b'][a]; slot = (column (k, b'), segment of a')
#pragma unroll
        for (int q = 0; q < XC; ++q) {
            const int w = threadIdx.x + q * NT;
            int col, sg;
            t3_slot<SG>(w, col, sg);
            if (w < nslot && col < nk * P) {
                R x[P];
#pragma unroll
                for (int a = 0; a < P; ++a) x[a] = T2[col * TS + a];
#pragma unroll
                for (int i = 0; i < PS; ++i)
                    if (sg * PS + i < P) acc[q][i] = row_dot(U0 + (sg * PS + i) * PR, x, acc[q][i]);
            }
        }
    }
    // [c' = k0 + k][b'][a'] is contiguous: through T1 (read last before the barrier above).  Stores of
    // a row a lane: N = 1e6 FP64, 4096 boxes, 205 us; through T1 166
#pragma unroll
    for (int q = 0; q < XC; ++q) {
        const int w = threadIdx.x + q * NT;
        int col, sg;
        t3_slot<SG>(w, col, sg);
        if (w < nslot && col < nk * P) {
#pragma unroll
            for (int i = 0; i < PS; ++i)
                if (sg * PS + i < P) T1[col * P + sg * PS + i] = acc[q][i];
        }
    }
    __syncthreads();
    R *dst = out + (size_t)k0 * PP;
    for (int i = threadIdx.x; i < nk * PP; i += NT) dst[i] = add ? dst[i] + T1[i] : T1[i];
}

// The same transform in FP32 at p = 18 on 4-wide matrix-core blocks (v_mfma_f32_4x4x1, see
// k_charge2proxy): a lane owns a column and supplies its input as the B operand, the matrix rows
// come as the A operand that broadcasts one block of 4 outputs to all lanes.  A workgroup of 6
// waves takes 9 of an item's 18 output planes: z in 6 column groups (12 outputs of 5 inputs fill
// an A register), y and x in 3 column groups x 2 parts of the outputs (20 outputs of 3 inputs).
// Every output is the chain of fused multiply-adds of k_tensor3 (c, b, a ascending, inputs in
// order), bit for bit.  The outputs leave through LDS: 12 scalar stores a lane, 72 bytes apart,
// held the kernel at the vector kernel's time.
// Alone, N = 1e6: 4096 items 142 -> 77 us (stores as scalars 142), 512 items 27 -> 14; what
// bounds it now is memory: 95 MB written and the products between the three barriers.
struct T3m4Cfg {
    static constexpr int P = 18, K = 9, NW = 6, TS = 19, slices = P / K;
};
template <int GPR, int G0, int C, int... I>
__device__ __forceinline__ void t3m4_step(float a, float x, c2p_f4 *acc, std::integer_sequence<int, I...>) {
    ((acc[I] = __builtin_amdgcn_mfma_f32_4x4x1f32(a, x, acc[I], 4, C % (16 / GPR) * GPR + G0 + I, 0)), ...);
}
// acc += outputs 4 G0 .. 4 (G0 + GN) - 1 of one column over its inputs; GPR groups of 4 outputs
// per input, 16 / GPR inputs per A register
template <int GPR, int G0, int GN, int... C>
__device__ __forceinline__ void t3m4_column(const float *a, const float *x, c2p_f4 *acc, std::integer_sequence<int, C...>) {
    (t3m4_step<GPR, G0, C>(a[C / (16 / GPR)], x[C], acc, std::make_integer_sequence<int, GN>{}), ...);
}
template <bool TRANSPOSE>
__global__ __launch_bounds__(64 * T3m4Cfg::NW, 2) void k_tensor3_m4(
    const float *__restrict__ in_base, float *__restrict__ out_base, const int *__restrict__ item_out,
    const int *__restrict__ item_add, const int *__restrict__ item_ptr, const int *__restrict__ in_slot,
    const int *__restrict__ in_code, const float *__restrict__ mats_rm, long long vs_in, long long vs_out) {
    chain_priority();
    in_base += (long long)blockIdx.z * vs_in;
    out_base += (long long)blockIdx.z * vs_out;
    constexpr int P = T3m4Cfg::P, K = T3m4Cfg::K, TS = T3m4Cfg::TS, PP = P * P, NC = K * P;
    static_assert(NC * P <= K * PP && NC * P % 4 == 0 && K * PP % 4 == 0, "output staging");
    __shared__ __align__(16) float T1[K * PP], T2[NC * TS];  // T1[k][b][a], T2[k][b'][a]
    const int lg = xcd_block(blockIdx.x, gridDim.x), it = lg / T3m4Cfg::slices, k0 = (lg % T3m4Cfg::slices) * K;
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const float *Ubase = mats_rm + (TRANSPOSE ? 2 : 0) * PP;
    float *out = out_base + (size_t)item_out[it] * P * PP;
    const bool add = item_add[it] != 0;
    const int e0 = item_ptr[it], e1 = item_ptr[it + 1];
    using Cs = std::make_integer_sequence<int, P>;
    // this wave's column of y and x (clamped to the last one), and its part of the outputs
    const int col = 64 * (w / 2) + lane, cc = min(col, NC - 1), kk = cc / P, aa = cc - kk * P;
    const bool low = w % 2 == 0;  // outputs 0 .. 11, else 12 .. 17
    // A registers of y and x: U(o, c), input c = 3 r + lane / 20, output o = lane % 20; of z: input
    // c = 5 r + lane / 12, output k0 + lane % 12
    const int ac = lane / 20, ao = lane % 20, zc = lane / 12, zo = lane % 12;
    c2p_f4 acc[3];
#pragma unroll
    for (int g = 0; g < 3; ++g) acc[g] = c2p_f4{0, 0, 0, 0};
    for (int e = e0; e < e1; ++e) {
        const float *in = in_base + (size_t)in_slot[e] * P * PP;
        const int code = in_code[e];
        const float *U0 = Ubase + (code & 1) * PP, *U1 = Ubase + ((code >> 1) & 1) * PP,
                    *U2 = Ubase + ((code >> 2) & 1) * PP;
        float az[4], a1[6], a0[6];
#pragma unroll
        for (int r = 0; r < 4; ++r) az[r] = zo < K && zc < 5 && 5 * r + zc < P ? U2[(k0 + zo) * P + 5 * r + zc] : 0.0f;
#pragma unroll
        for (int r = 0; r < 6; ++r) {
            const bool in_u = ao < P && ac < 3;
            a1[r] = in_u ? U1[ao * P + 3 * r + ac] : 0.0f;
            a0[r] = in_u ? U0[ao * P + 3 * r + ac] : 0.0f;
        }
        // z: T1[k][b][a] = sum_c U2(k0 + k, c) in[c][b][a].  (T1's last readers are a barrier back.)
        {
            const int j = 64 * w + lane, jc = min(j, PP - 1);
            float x[P];
#pragma unroll
            for (int c = 0; c < P; ++c) x[c] = in[c * PP + jc];
            c2p_f4 z[3];
#pragma unroll
            for (int g = 0; g < 3; ++g) z[g] = c2p_f4{0, 0, 0, 0};
            t3m4_column<3, 0, 3>(az, x, z, Cs{});
            if (j < PP)
#pragma unroll
                for (int k = 0; k < K; ++k) T1[k * PP + j] = z[k >> 2][k & 3];
        }
        __syncthreads();
        // y: T2[k][b'][a] = sum_b U1(b', b) T1[k][b][a]
        {
            float x[P];
#pragma unroll
            for (int b = 0; b < P; ++b) x[b] = T1[kk * PP + b * P + aa];
            c2p_f4 y[3];
#pragma unroll
            for (int g = 0; g < 3; ++g) y[g] = c2p_f4{0, 0, 0, 0};
            if (low) t3m4_column<5, 0, 3>(a1, x, y, Cs{});
            else t3m4_column<5, 3, 2>(a1, x, y, Cs{});
            float *dst = T2 + (size_t)(kk * P + (low ? 0 : 12)) * TS + aa;
            if (col < NC)
#pragma unroll
                for (int i = 0; i < 12; ++i)
                    if (i < 6 || low) dst[i * TS] = y[i >> 2][i & 3];
        }
        __syncthreads();
        // x: acc[a'] += sum_a U0(a', a) T2[k][b'][a]
        {
            float x[P];
#pragma unroll
            for (int a = 0; a < P; ++a) x[a] = T2[cc * TS + a];
            if (low) t3m4_column<5, 0, 3>(a0, x, acc, Cs{});
            else t3m4_column<5, 3, 2>(a0, x, acc, Cs{});
        }
    }
    // [c' = k0 + k][b'][a'] is contiguous: through T1 (read last before the barrier above), 16 bytes a lane
    if (col < NC)
#pragma unroll
        for (int i = 0; i < 12; ++i)
            if (i < 6 || low) T1[col * P + (low ? 0 : 12) + i] = acc[i >> 2][i & 3];
    __syncthreads();
    float4 *dst = reinterpret_cast<float4 *>(out + (size_t)k0 * PP);
    for (int i = threadIdx.x; i < NC * P / 4; i += 64 * T3m4Cfg::NW) {
        float4 v = reinterpret_cast<const float4 *>(T1)[i];
        if (add) {
            const float4 o = dst[i];
            v.x = o.x + v.x, v.y = o.y + v.y, v.z = o.z + v.z, v.w = o.w + v.w;
        }
        dst[i] = v;
    }
}

// The same transform for FP64 at p = 28 on the matrix cores (v_mfma_f64_16x16x4f64,
// operand and accumulator layout as in k_eval_targets_mfma).  Workgroup (item, ct) computes
// the output planes c' in [16 ct, 16 ct + 16), the item's inputs taken in slices of 4 values
// of a:
//   z:  T1[c'][(b, al)]  = sum_c U2(c', c) in[c][b][4 s + al]        (16 rows, 4 p columns)
//   y:  T2[(c', b')][al] = sum_b U1(b', b) T1[c'][(b, al)]            (rows b', 64 columns)
//   x:  out[(c', b')][a'] += sum_al U0(a', 4 s + al) T2[(c', b')][al] (rows a', 16 p columns)
// z and y go through LDS, x into accumulators that persist over the slices and the item's
// inputs (a wave owns x's column tiles w, w + NW, ...).  Every output sums its terms in the
// order of k_tensor3 (c, then b, then a ascending, inputs in order), so the two kernels agree
// to the last bit.  LDS holds both matrices transposed (Ut[c][r], zero-padded, so fragment
// reads need no bounds checks) and the two slice buffers (zero where c' or b is past p).
template <int P> struct T3MfmaCfg {
    static constexpr int PP = P * P;
    static constexpr int KS = (P + 3) / 4;        // 4-steps of a contraction = slices of a
    static constexpr int CT = (P + 15) / 16;      // 16-row tiles of an output index
    static constexpr int NW = P >= 38 ? 8 : 4;    // waves per workgroup
    static constexpr int XT = (P + NW - 1) / NW;  // x column tiles per wave (16 p columns = p tiles)
    static constexpr int LP = 16 * CT + 8;        // row stride of Ut (8 mod 16: a fragment's rows
    static constexpr int S1 = 16 * KS + 8;        // and those of T1 fall on different banks)
};

template <int P, bool TRANSPOSE>
__global__ __launch_bounds__(64 * T3MfmaCfg<P>::NW) void k_tensor3_mfma(
    const double *__restrict__ in_base, double *__restrict__ out_base, const int *__restrict__ item_out,
    const int *__restrict__ item_add, const int *__restrict__ item_ptr, const int *__restrict__ in_slot,
    const int *__restrict__ in_code, const double *__restrict__ mats_rm, int n_items, long long vs_in = 0,
    long long vs_out = 0) {
    chain_priority();
    in_base += (long long)blockIdx.z * vs_in;  // vector blockIdx.z of a many-vector launch
    out_base += (long long)blockIdx.z * vs_out;
    using Cfg = T3MfmaCfg<P>;
    using M = Mfma16<double>;
    typedef M::acc_t acc_t;
    constexpr int PP = Cfg::PP, KS = Cfg::KS, CT = Cfg::CT, NW = Cfg::NW, XT = Cfg::XT, LP = Cfg::LP, S1 = Cfg::S1,
                  NT = 64 * NW;
    __shared__ double Ut[2 * 4 * KS * LP];  // Ut[s][c][r] = U_s(r, c), zero outside r, c < p
    __shared__ double T1[16 * S1];          // [c' - 16 ct][(b, al)]
    __shared__ double T2[16 * P * 4];       // [(c' - 16 ct, b')][al]
    const int lg = xcd_block(blockIdx.x, gridDim.x), it = lg / CT, ct = lg - it * CT;
    if (it >= n_items) return;
    const double *Ubase = mats_rm + (TRANSPOSE ? 2 : 0) * PP;
    for (int i = threadIdx.x; i < 2 * 4 * KS * LP; i += NT) {
        const int sd = i / (4 * KS * LP), c = (i / LP) % (4 * KS), r = i % LP;
        Ut[i] = (r < P && c < P) ? Ubase[sd * PP + r * P + c] : 0.0;
    }
    for (int i = threadIdx.x; i < 16 * S1; i += NT) T1[i] = 0.0;
    for (int i = threadIdx.x; i < 16 * P * 4; i += NT) T2[i] = 0.0;
    const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), l = threadIdx.x & 63, kk = l >> 4,
              jj = l & 15;
    acc_t acc[XT][CT];
#pragma unroll
    for (int t = 0; t < XT; ++t)
#pragma unroll
        for (int mt = 0; mt < CT; ++mt) acc[t][mt] = acc_t{0.0, 0.0, 0.0, 0.0};
    const int e0 = item_ptr[it], e1 = item_ptr[it + 1];
    for (int e = e0; e < e1; ++e) {
        const double *in = in_base + (size_t)in_slot[e] * P * PP;
        const int code = in_code[e];
        const double *U0 = Ut + (code & 1) * 4 * KS * LP, *U1 = Ut + ((code >> 1) & 1) * 4 * KS * LP,
                     *U2 = Ut + ((code >> 2) & 1) * 4 * KS * LP;
        for (int s = 0; s < KS; ++s) {
            __syncthreads();  // Ut and the zero padding written; the previous y done with T1
            // z: one job per 16 columns (b, al)
            for (int nt = w; nt < KS; nt += NW) {
                const int n = 16 * nt + jj, b = n >> 2, a = 4 * s + (n & 3);
                acc_t d = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
                for (int ks = 0; ks < KS; ++ks) {
                    const int c = 4 * ks + kk;
                    const double bv = (c < P && b < P && a < P) ? in[(size_t)c * PP + b * P + a] : 0.0;
                    d = M::mma(U2[c * LP + 16 * ct + jj], bv, d);
                }
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int cl = M::row(kk, q);
                    if (16 * ct + cl < P && b < P) T1[cl * S1 + n] = d[q];
                }
            }
            __syncthreads();
            // y: job = (row tile of b', one of the 4 column tiles of (c', al))
            for (int job = w; job < 4 * CT; job += NW) {
                const int mt = job % CT, nt = job / CT;
                const int n = 16 * nt + jj, cl = n >> 2, al = n & 3;
                acc_t d = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
                for (int ks = 0; ks < KS; ++ks) {
                    const int b = 4 * ks + kk;
                    d = M::mma(U1[b * LP + 16 * mt + jj], T1[cl * S1 + 4 * b + al], d);
                }
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int bp = 16 * mt + M::row(kk, q);
                    if (bp < P && 16 * ct + cl < P) T2[(cl * P + bp) * 4 + al] = d[q];
                }
            }
            __syncthreads();
            // x: this wave's column tiles of (c', b'), one 4-step over a = 4 s + al
#pragma unroll
            for (int t = 0; t < XT; ++t) {
                const int nt = w + NW * t;
                if (nt < P) {
                    const double bv = T2[(16 * nt + jj) * 4 + kk];
#pragma unroll
                    for (int mt = 0; mt < CT; ++mt)
                        acc[t][mt] = M::mma(U0[(4 * s + kk) * LP + 16 * mt + jj], bv, acc[t][mt]);
                }
            }
        }
    }
    double *out = out_base + (size_t)item_out[it] * P * PP + (size_t)16 * ct * PP;
    const bool add = item_add[it] != 0;
#pragma unroll
    for (int t = 0; t < XT; ++t) {
        const int n = 16 * (w + NW * t) + jj;  // (c' - 16 ct) p + b'
        if (w + NW * t >= P || 16 * ct + n / P >= P) continue;
#pragma unroll
        for (int mt = 0; mt < CT; ++mt)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int ap = 16 * mt + M::row(kk, q);
                if (ap < P) {
                    double *dst = out + (size_t)n * P + ap;
                    *dst = add ? *dst + acc[t][mt][q] : acc[t][mt][q];
                }
            }
    }
}

// proxy[parent_slot[i]] += sum_{k in child_ptr[i] .. child_ptr[i+1]} scratch[k], element-wise, the
// children added in order (deterministic).
template <class R, int P>
__global__ __launch_bounds__(256) void k_sum_children(R *__restrict__ proxy, const R *__restrict__ scratch,
                                                       const int *__restrict__ parent_slot, const int *__restrict__ child_ptr,
                                                       int n_parents, long long vs_proxy = 0, long long vs_scratch = 0) {
    chain_priority();
    proxy += (long long)blockIdx.z * vs_proxy;  // vector blockIdx.z of a many-vector launch
    scratch += (long long)blockIdx.z * vs_scratch;
    constexpr int P3 = P * P * P;
    const int it = blockIdx.x, e = blockIdx.y * blockDim.x + threadIdx.x;
    if (it >= n_parents || e >= P3) return;
    R *dst = proxy + (size_t)parent_slot[it] * P3 + e;
    R v = *dst;
    for (int k = child_ptr[it]; k < child_ptr[it + 1]; ++k) v += scratch[(size_t)k * P3 + e];
    *dst = v;
}

// ------------------------------------------------------------------ plane waves
// Plane-wave mode layout: m = k1 * (H n) + k3 * n + k2 ([x][z][y], y fastest), k3 < H.
// The polynomial <-> plane-wave matrices have the parity of the Chebyshev polynomials:
// W(k, j) = sum_i Vinv(j, i) e^{-i (k - n/2) x_i h} over nodes x_i symmetric about 0 with
// T_j(-x) = (-1)^j T_j(x), so W(k, j) is real for even j and imaginary for odd j (the other
// part is rounding, below 1e-15 of the largest entry).  The transforms use that: a product
// with W(k, j) costs one real multiply-add per real component instead of two.
// Outgoing expansion pw(k1,k2,k3) = sum W(k1,a) W(k2,b) W(k3,c) C[c][b][a], W = poly2pw
// (W(k, j) at W[k + n j]); one workgroup per (box, slice of k3), 1-D grid, (box, slice) at
// xcd_block index box * slices + slice (a box's slices share one L2).  Box x reads proxy
// slot slot0 + x and writes plane-wave slot x.
// The z step of whole boxes into HBM, for orders where the slices of k_proxy2pw would each
// re-read the box's proxy charges (20 slices per box for FP64 at p = 28, 28 at p = 38):
// t1[box][k][b][a] = sum_c W(k, c) C[c][b][a] for k < H, one thread per column (b, a), the
// same sums as k_proxy2pw's z step.  k_p2pw_yx then takes each plane of t1 through the y and
// x steps.
template <class R, int P, int NPW>
__global__ __launch_bounds__(256) void k_p2pw_z(const R *__restrict__ proxy, Cx<R> *__restrict__ t1,
                                                const Cx<R> *__restrict__ W, int slot0, int n_boxes) {
    chain_priority();
    constexpr int H = (NPW + 1) / 2, PP = P * P, PER = (PP + 255) / 256;  // workgroups per box
    const int lg = xcd_block(blockIdx.x, gridDim.x), bx = lg / PER, j = (lg - bx * PER) * 256 + (int)threadIdx.x;
    if (bx >= n_boxes || j >= PP) return;
    const R *C = proxy + (size_t)(slot0 + bx) * P * PP;
    Cx<R> *out = t1 + (size_t)bx * H * PP;
    R x[P];
#pragma unroll
    for (int c = 0; c < P; ++c) x[c] = C[c * PP + j];
    for (int k = 0; k < H; ++k) {
        R sr = 0, si = 0;
#pragma unroll
        for (int c = 0; c < P; c += 2) sr = fma(W[k + NPW * c].re, x[c], sr);
#pragma unroll
        for (int c = 1; c < P; c += 2) si = fma(W[k + NPW * c].im, x[c], si);
        out[(size_t)k * PP + j] = {sr, si};
    }
}

template <class R, int P, int NPW, int BK = 0>
__global__ __launch_bounds__(256) void k_proxy2pw(const R *__restrict__ proxy, Cx<R> *__restrict__ pw_out,
                                                   const Cx<R> *__restrict__ W, int slot0, int n_boxes,
                                                   long long vs_in = 0, long long vs_out = 0) {
    chain_priority();
    proxy += (long long)blockIdx.z * vs_in;  // vector blockIdx.z of a many-vector launch
    pw_out += (long long)blockIdx.z * vs_out;
    constexpr int H = (NPW + 1) / 2, COL = H * NPW, PP = P * P, TS = OddStride<P>::v;
    constexpr int K3 = P2pwCfg<R, P, NPW, BK>::K3;
    __shared__ Cx<R> T1[K3 * PP];        // [k][b][a]
    __shared__ Cx<R> T2[K3 * NPW * TS];  // [k][k2][a] rows of TS
    constexpr int NS = P2pwCfg<R, P, NPW, BK>::slices;
    const int lg = xcd_block(blockIdx.x, gridDim.x), bx = lg / NS, slice = lg - bx * NS;
    if (bx >= n_boxes) return;
    const R *C = proxy + (size_t)(slot0 + bx) * P * PP;
    Cx<R> *pw = pw_out + (size_t)bx * NPW * COL;
    {
        const int k30 = slice * K3;  // this workgroup's slice of k3
        const int nk = min(K3, H - k30);
        // z: T1[k][b][a] = sum_c W(k30 + k, c) C[c][b][a]
        for (int j = threadIdx.x; j < PP; j += blockDim.x) {
            R x[P];
#pragma unroll
            for (int c = 0; c < P; ++c) x[c] = C[c * PP + j];
            for (int k = 0; k < nk; ++k) {
                R sr = 0, si = 0;
#pragma unroll
                for (int c = 0; c < P; c += 2) sr = fma(W[k30 + k + NPW * c].re, x[c], sr);
#pragma unroll
                for (int c = 1; c < P; c += 2) si = fma(W[k30 + k + NPW * c].im, x[c], si);
                T1[k * PP + j] = {sr, si};
            }
        }
        __syncthreads();
        // y: T2[k][k2][a] = sum_b W(k2, b) T1[k][b][a]; slot = (column (k, a), segment of k2,
        // uniform across a wavefront)
        constexpr int SGY = P2pwCfg<R, P, NPW, BK>::SGY, PSY = P2pwCfg<R, P, NPW, BK>::PSY;
        const int ny = (nk * P + 63) / 64 * 64 * SGY;
        for (int t = threadIdx.x; t < ny; t += blockDim.x) {
            int w, sg;
            t3_slot<SGY>(t, w, sg);
            if (w >= nk * P) continue;
            const int k = w / P, a = w - k * P;
            Cx<R> v[P];
#pragma unroll
            for (int b = 0; b < P; ++b) v[b] = T1[k * PP + b * P + a];
            for (int k2 = sg * PSY; k2 < min(NPW, sg * PSY + PSY); ++k2) {
                R sr = 0, si = 0;
#pragma unroll
                for (int b = 0; b < P; ++b) {
                    if (b % 2 == 0) {
                        const R m = W[k2 + NPW * b].re;
                        sr = fma(m, v[b].re, sr);
                        si = fma(m, v[b].im, si);
                    } else {
                        const R m = W[k2 + NPW * b].im;
                        sr = fma(-m, v[b].im, sr);
                        si = fma(m, v[b].re, si);
                    }
                }
                T2[(k * NPW + k2) * TS + a] = {sr, si};
            }
        }
        __syncthreads();
        // x: pw[k1][k30 + k][k2] = sum_a W(k1, a) T2[k][k2][a]; slot = (column w = k n + k2,
        // segment of k1, uniform across a wavefront)
        constexpr int SGX = P2pwCfg<R, P, NPW, BK>::SGX, PSX = P2pwCfg<R, P, NPW, BK>::PSX;
        const int nx = (nk * NPW + 63) / 64 * 64 * SGX;
        for (int t = threadIdx.x; t < nx; t += blockDim.x) {
            int w, sg;
            t3_slot<SGX>(t, w, sg);
            if (w >= nk * NPW) continue;
            Cx<R> v[P];
#pragma unroll
            for (int a = 0; a < P; ++a) v[a] = T2[w * TS + a];
            Cx<R> *dst = pw + (size_t)k30 * NPW + w;
            for (int k1 = sg * PSX; k1 < min(NPW, sg * PSX + PSX); ++k1) {
                R sr = 0, si = 0;
#pragma unroll
                for (int a = 0; a < P; ++a) {
                    if (a % 2 == 0) {
                        const R m = W[k1 + NPW * a].re;
                        sr = fma(m, v[a].re, sr);
                        si = fma(m, v[a].im, si);
                    } else {
                        const R m = W[k1 + NPW * a].im;
                        sr = fma(-m, v[a].im, sr);
                        si = fma(m, v[a].re, si);
                    }
                }
                dst[(size_t)k1 * COL] = {sr, si};
            }
        }
    }
}

// The same transform in FP32 at p = 18 (n = 27) on 4-wide matrix-core blocks (v_mfma_f32_4x4x1, see
// k_charge2proxy): a lane owns a column and supplies its input as the B operand, the folded
// matrix F[j][k] (real part of W(k, j) for even j, imaginary part for odd j) comes as the A operand
// that broadcasts one block of 4 outputs to all lanes; 28 outputs of two j fill one register.
// The parity of j picks the components as in k_proxy2pw, and every output is the same chain of
// fused multiply-adds over j, bit for bit.  A workgroup of 6 waves takes 7 k3 planes of a box
// (half the box): z in 6 column groups, y in 2 groups x 3 parts of the outputs, x in 3 x 2.
// The vector kernel ran at 29% of the vector rate on its matrix loads; 432 boxes x 4 vectors:
// 106 -> 54 us, 576 boxes 36 -> 22 us, 64 boxes 11.5 -> 5.4 us alone.
struct P2pw4Cfg {
    static constexpr int P = 18, NPW = 27, H = 14, K3 = 7, KG = 7, NW = 6, TS = 19, slices = H / K3;
};
template <int B, int G0, int... I>
__device__ __forceinline__ void p2pw4_step(float a, Cx<float> v, c2p_f4 *re, c2p_f4 *im, std::integer_sequence<int, I...>) {
    const float xr = (B & 1) ? -v.im : v.re, xi = (B & 1) ? v.re : v.im;
    constexpr int blk = (B & 1) * P2pw4Cfg::KG + G0;
    ((re[I] = __builtin_amdgcn_mfma_f32_4x4x1f32(a, xr, re[I], 4, blk + I, 0)), ...);
    ((im[I] = __builtin_amdgcn_mfma_f32_4x4x1f32(a, xi, im[I], 4, blk + I, 0)), ...);
}
// outputs 4 G0 .. 4 (G0 + GN) - 1 of one column over its 18 inputs
template <int G0, int GN, int... B>
__device__ __forceinline__ void p2pw4_column(const float *a, const Cx<float> *v, c2p_f4 *re, c2p_f4 *im,
                                             std::integer_sequence<int, B...>) {
#pragma unroll
    for (int g = 0; g < GN; ++g) re[g] = im[g] = c2p_f4{0, 0, 0, 0};
    (p2pw4_step<B, G0>(a[B / 2], v[B], re, im, std::make_integer_sequence<int, GN>{}), ...);
}
template <int... C>
__device__ __forceinline__ void p2pw4_z(const float *a, const float *x, c2p_f4 *re, c2p_f4 *im, std::integer_sequence<int, C...>) {
    // even c into re, odd c into im, outputs in 2 groups
    (((C & 1) ? (im[0] = __builtin_amdgcn_mfma_f32_4x4x1f32(a[C / 8], x[C], im[0], 4, C % 8 * 2, 0),
                 im[1] = __builtin_amdgcn_mfma_f32_4x4x1f32(a[C / 8], x[C], im[1], 4, C % 8 * 2 + 1, 0))
              : (re[0] = __builtin_amdgcn_mfma_f32_4x4x1f32(a[C / 8], x[C], re[0], 4, C % 8 * 2, 0),
                 re[1] = __builtin_amdgcn_mfma_f32_4x4x1f32(a[C / 8], x[C], re[1], 4, C % 8 * 2 + 1, 0))),
     ...);
}
__global__ __launch_bounds__(64 * P2pw4Cfg::NW, 2) void k_proxy2pw_m4(const float *__restrict__ proxy,
                                                                      Cx<float> *__restrict__ pw_out,
                                                                      const float *__restrict__ F, int slot0,
                                                                      long long vs_in, long long vs_out) {
    chain_priority();
    proxy += (long long)blockIdx.z * vs_in;
    pw_out += (long long)blockIdx.z * vs_out;
    constexpr int P = P2pw4Cfg::P, NPW = P2pw4Cfg::NPW, H = P2pw4Cfg::H, K3 = P2pw4Cfg::K3, TS = P2pw4Cfg::TS, PP = P * P,
                  COL = H * NPW, NS = P2pw4Cfg::slices;
    __shared__ Cx<float> T1[K3 * PP], T2[K3 * NPW * TS];
    const int lg = xcd_block(blockIdx.x, gridDim.x), bx = lg / NS, k30 = (lg - bx * NS) * K3;
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const float *C = proxy + (size_t)(slot0 + bx) * P * PP;
    using Js = std::make_integer_sequence<int, P>;
    // A registers: rows 2 r and 2 r + 1 of F, 28 outputs each; for z rows 8 r .. 8 r + 7, this
    // workgroup's 7 outputs (and one more) each
    float a[P / 2], az[3];
#pragma unroll
    for (int r = 0; r < P / 2; ++r) a[r] = lane < 56 ? F[(2 * r + (lane >= 28)) * 64 + lane - (lane >= 28 ? 28 : 0)] : 0.0f;
#pragma unroll
    for (int r = 0; r < 3; ++r) {
        const int j = 8 * r + lane / 8;
        az[r] = j < P ? F[j * 64 + k30 + lane % 8] : 0.0f;
    }
    {
        const int col = 64 * w + lane, cc = min(col, PP - 1);
        float x[P];
#pragma unroll
        for (int c = 0; c < P; ++c) x[c] = C[c * PP + cc];
        c2p_f4 re[2], im[2];
#pragma unroll
        for (int g = 0; g < 2; ++g) re[g] = im[g] = c2p_f4{0, 0, 0, 0};
        p2pw4_z(az, x, re, im, Js{});
        if (col < PP)
#pragma unroll
            for (int k = 0; k < K3; ++k) T1[k * PP + col] = {re[k >> 2][k & 3], im[k >> 2][k & 3]};
    }
    __syncthreads();
    {
        const int col = 64 * (w / 3) + lane, cc = min(col, K3 * P - 1), k = cc / P, aa = cc - k * P;
        Cx<float> v[P];
#pragma unroll
        for (int b = 0; b < P; ++b) v[b] = T1[k * PP + b * P + aa];
        auto part = [&](auto g0, auto gn) {
            constexpr int G0 = decltype(g0)::value, GN = decltype(gn)::value;
            c2p_f4 re[GN], im[GN];
            p2pw4_column<G0, GN>(a, v, re, im, Js{});
            if (col < K3 * P)
#pragma unroll
                for (int i = 0; i < 4 * GN; ++i)
                    if (4 * G0 + i < NPW) T2[(k * NPW + 4 * G0 + i) * TS + aa] = {re[i >> 2][i & 3], im[i >> 2][i & 3]};
        };
        const int sub = w % 3;
        if (sub == 0) part(std::integral_constant<int, 0>{}, std::integral_constant<int, 3>{});
        else if (sub == 1) part(std::integral_constant<int, 3>{}, std::integral_constant<int, 2>{});
        else part(std::integral_constant<int, 5>{}, std::integral_constant<int, 2>{});
    }
    __syncthreads();
    {
        const int col = 64 * (w / 2) + lane, cc = min(col, K3 * NPW - 1);
        Cx<float> v[P];
#pragma unroll
        for (int i = 0; i < P; ++i) v[i] = T2[cc * TS + i];
        Cx<float> *dst = pw_out + (size_t)bx * NPW * COL + (size_t)k30 * NPW + cc;
        auto part = [&](auto g0, auto gn) {
            constexpr int G0 = decltype(g0)::value, GN = decltype(gn)::value;
            c2p_f4 re[GN], im[GN];
            p2pw4_column<G0, GN>(a, v, re, im, Js{});
            if (col < K3 * NPW)
#pragma unroll
                for (int i = 0; i < 4 * GN; ++i)
                    if (4 * G0 + i < NPW) dst[(size_t)(4 * G0 + i) * COL] = {re[i >> 2][i & 3], im[i >> 2][i & 3]};
        };
        if (w % 2 == 0) part(std::integral_constant<int, 0>{}, std::integral_constant<int, 4>{});
        else part(std::integral_constant<int, 4>{}, std::integral_constant<int, 3>{});
    }
}

// Incoming expansion of one level: pin[i][m] = lscale sum_e pw_out[slot_e - slot0][m] shift0[sten_e][m]
// over box i's CSR range of (neighbour slot, stencil); shift0 holds the level-0 translation
// times the radial Fourier factor, lscale = 2^level scales the latter to this level.
template <class R>
__global__ __launch_bounds__(256) void k_pw_shift(const Cx<R> *__restrict__ pw_out, const Cx<R> *__restrict__ shift0,
                                                   R lscale, const int *__restrict__ nbr_ptr,
                                                   const int *__restrict__ nbr_slot, const int *__restrict__ nbr_sten,
                                                   int slot0, int nm, int item0, Cx<R> *__restrict__ pin,
                                                   long long vs_in = 0, long long vs_out = 0) {
    chain_priority();
    pw_out += (long long)blockIdx.z * vs_in;  // vector blockIdx.z of a many-vector launch
    pin += (long long)blockIdx.z * vs_out;
    // x = target box (consecutive workgroups share neighbours; each XCD takes a contiguous,
    // spatially coherent range of boxes), y = mode chunk: the neighbours' chunk is read from
    // L2 by the 27 boxes around it instead of from memory
    const int bi = xcd_block(blockIdx.x, gridDim.x), it = item0 + bi;
    const int m = blockIdx.y * blockDim.x + threadIdx.x;
    if (m >= nm) return;
    R sr = 0, si = 0;
    for (int e = nbr_ptr[it]; e < nbr_ptr[it + 1]; ++e) {
        const Cx<R> a = pw_out[(size_t)(nbr_slot[e] - slot0) * nm + m];
        const Cx<R> s = shift0[(size_t)nbr_sten[e] * nm + m];
        sr = fma(a.re, s.re, fma(-a.im, s.im, sr));
        si = fma(a.re, s.im, fma(a.im, s.re, si));
    }
    pin[(size_t)bi * nm + m] = {sr * lscale, si * lscale};
}

// The same sum in FP64 with the shift factors formed from their separable parts instead of
// read from the 27-stencil table (27 n^2 h complex values, 13 MB at p = 28, more than an XCD's
// L2, so every target box's shifts streamed it from memory beside the neighbours' plane
// waves): shift0[t][m] = radial0[m] e^{i (x_c dx + x_a dz + x_b dy)} for the mode
// m = (c h + a) n + b and stencil t = 9 (dz + 1) + 3 (dy + 1) + (dx + 1), x_j = (j - n/2) sphase;
// ephase[j] = e^{i x_j}, taken conjugated for an offset of -1 and left out for 0.  The radial
// factor multiplies the sum once.
__global__ __launch_bounds__(256) void k_pw_shift_sep(const Cx<double> *__restrict__ pw_out,
                                                      const double *__restrict__ radial0,
                                                      const Cx<double> *__restrict__ ephase, double lscale,
                                                      const int *__restrict__ nbr_ptr, const int *__restrict__ nbr_slot,
                                                      const int *__restrict__ nbr_sten, int slot0, int nm, int item0,
                                                      int n, int h, Cx<double> *__restrict__ pin, long long vs_in = 0,
                                                      long long vs_out = 0) {
    chain_priority();
    pw_out += (long long)blockIdx.z * vs_in;  // vector blockIdx.z of a many-vector launch
    pin += (long long)blockIdx.z * vs_out;
    const int bi = xcd_block(blockIdx.x, gridDim.x), it = item0 + bi;
    const int m = blockIdx.y * blockDim.x + threadIdx.x;
    if (m >= nm) return;
    const int b = m % n, a = (m / n) % h, c = m / (n * h);
    const Cx<double> ex = ephase[c], ez = ephase[a], ey = ephase[b];
    double sr = 0, si = 0;
    for (int e = nbr_ptr[it]; e < nbr_ptr[it + 1]; ++e) {
        const int t = nbr_sten[e], dz = t / 9 - 1, dy = (t / 3) % 3 - 1, dx = t % 3 - 1;  // uniform
        double fr = 1, fi = 0;
        if (dz) {
            fr = ez.re;
            fi = dz > 0 ? ez.im : -ez.im;
        }
        if (dy) {
            const double gi = dy > 0 ? ey.im : -ey.im, r = fr * ey.re - fi * gi;
            fi = fma(fr, gi, fi * ey.re);
            fr = r;
        }
        if (dx) {
            const double gi = dx > 0 ? ex.im : -ex.im, r = fr * ex.re - fi * gi;
            fi = fma(fr, gi, fi * ex.re);
            fr = r;
        }
        const Cx<double> av = pw_out[(size_t)(nbr_slot[e] - slot0) * nm + m];
        sr = fma(av.re, fr, fma(-av.im, fi, sr));
        si = fma(av.re, fi, fma(av.im, fr, si));
    }
    const double rr = radial0[m] * lscale;
    pin[(size_t)bi * nm + m] = {sr * rr, si * rr};
}

// Folded matrix table of the plane-wave transforms: F[j * 64 + k] = W(k, j).re for even j,
// W(k, j).im for odd j (the entry's only non-zero part), 0 for k >= n; k in a row of 64.
//
// Second pass of the two-pass proxy -> plane-wave transform (after k_p2pw_z), FP64 on the
// matrix cores: the y and x steps of one k3 plane per wavefront.  With the parity folded into
// the operands, each step is a pair of real products with F:
//   y:  T2t[a][k2] = sum_b X[b][a] F[b][k2],  X = (T.re, T.im) for even b, (-T.im, T.re) for odd b
//   x:  pw[k1][k2] = sum_a F[a][k1] Z[a][k2], Z = (T2.re, T2.im) for even a, (-T2.im, T2.re) odd a
// (T[b][a] = the plane of t1).  v_mfma_f64_16x16x4f64 leaves y's output tile with lane l
// holding rows a = 4 e + l/16 of column l%16, which is the B operand x needs for the
// 4-row steps e = 0..3 of that tile, so the plane goes from y to x in registers, one 16-column
// tile of k2 at a time.  F sits in LDS (A and B fragments of both steps); the plane's t1 is
// read once per wavefront into registers.  Each output sums its terms in the same order as
// k_proxy2pw (b, then a, ascending).
template <int P, int NPW>
__global__ __launch_bounds__(256, 2) void k_p2pw_yx(const Cx<double> *__restrict__ t1, const double *__restrict__ F,
                                                 Cx<double> *__restrict__ pw_out, int n_boxes) {
    chain_priority();
    static_assert(NPW <= 64, "k2 and k1 within a table row of 64");
    using M = Mfma16<double>;
    typedef M::acc_t acc_t;
    constexpr int H = (NPW + 1) / 2, COL = H * NPW, PP = P * P, PG = (H + 3) / 4;  // 4 planes per workgroup
    constexpr int KS = (P + 3) / 4, AT = (P + 15) / 16, CT = (NPW + 15) / 16;     // 4-steps, a tiles, k tiles
    __shared__ double Fs[4 * KS * 64];
    for (int i = threadIdx.x; i < 4 * KS * 64; i += 256) Fs[i] = i < P * 64 ? F[i] : 0.0;
    __syncthreads();
    const int lg = xcd_block(blockIdx.x, gridDim.x), bx = lg / PG;
    const int k = (lg - bx * PG) * 4 + __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    if (bx >= n_boxes || k >= H) return;
    const int l = threadIdx.x & 63, kk = l >> 4, jj = l & 15;
    const bool odd = kk & 1;  // parity of b = 4 ks + kk (y) and of a = 16 at + 4 e + kk (x)
    const Cx<double> *T = t1 + ((size_t)bx * H + k) * PP;
    // y's A fragments: X[b = 4 ks + kk][a = 16 at + jj], real-output and imaginary-output parts
    double xr[KS][AT], xi[KS][AT];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
        for (int at = 0; at < AT; ++at) {
            const int b = 4 * ks + kk, a = 16 * at + jj;
            Cx<double> x = {0.0, 0.0};
            if (b < P && a < P) x = T[b * P + a];
            xr[ks][at] = odd ? -x.im : x.re;
            xi[ks][at] = odd ? x.re : x.im;
        }
    Cx<double> *dst = pw_out + (size_t)bx * NPW * COL + (size_t)k * NPW;
    // one k2 tile at a time (unrolled, the tiles' accumulators would take the registers of a
    // second wavefront per SIMD at p = 38)
#pragma unroll 1
    for (int ct = 0; ct < CT; ++ct) {  // k2 tile
        acc_t yr[AT], yi[AT];
#pragma unroll
        for (int at = 0; at < AT; ++at) yr[at] = yi[at] = acc_t{0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            const double f = Fs[(4 * ks + kk) * 64 + 16 * ct + jj];  // B[b][k2] = F[b][k2]
#pragma unroll
            for (int at = 0; at < AT; ++at) {
                yr[at] = M::mma(xr[ks][at], f, yr[at]);
                yi[at] = M::mma(xi[ks][at], f, yi[at]);
            }
        }
        // yr/yi[at][e] = T2 (re, im) at a = 16 at + 4 e + kk, k2 = 16 ct + jj: fold into Z
#pragma unroll
        for (int at = 0; at < AT; ++at)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const double re = yr[at][e], im = yi[at][e];
                yr[at][e] = odd ? -im : re;
                yi[at][e] = odd ? re : im;
            }
        for (int mt = 0; mt < CT; ++mt) {  // k1 tile
            acc_t pr = {0.0, 0.0, 0.0, 0.0}, pi = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int at = 0; at < AT; ++at)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    if (4 * at + e < KS) {
                        const double fa = Fs[(4 * (4 * at + e) + kk) * 64 + 16 * mt + jj];  // A[k1][a] = F[a][k1]
                        pr = M::mma(fa, yr[at][e], pr);
                        pi = M::mma(fa, yi[at][e], pi);
                    }
                }
            const int k2 = 16 * ct + jj;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int k1 = 16 * mt + M::row(kk, e);
                if (k1 < NPW && k2 < NPW) dst[(size_t)k1 * COL + k2] = {pr[e], pi[e]};
            }
        }
    }
}

// Shifts of groups of kShiftGroup consecutive target boxes (siblings, mostly): the group's
// neighbour lists merged by source slot, so each neighbour's plane waves are read once for
// the whole group (a 2x2x2 group of boxes has 64 distinct neighbours instead of 8 x 27).
// Entry e of group g: source slot gslot[e], and for target t of the group the stencil in
// byte t of gsten[e] (255: not a neighbour of t).  The shift factor comes from the
// 27-stencil table (FP32) or from the separable phases (FP64, as k_pw_shift_sep).  Targets
// sum their neighbours in slot order.
constexpr int kShiftGroup = 8;
template <class R>
__global__ __launch_bounds__(256) void k_pw_shift_grp(const Cx<R> *__restrict__ pw_out, const Cx<R> *__restrict__ shift0,
                                                      const double *__restrict__ radial0,
                                                      const Cx<double> *__restrict__ ephase, R lscale,
                                                      const int *__restrict__ gptr, const int *__restrict__ gslot,
                                                      const unsigned long long *__restrict__ gsten, int slot0, int nm,
                                                      int item0, int n_items, int n, int h, Cx<R> *__restrict__ pin,
                                                      long long vs_in = 0, long long vs_out = 0) {
    chain_priority();
    constexpr int G = kShiftGroup;
    pw_out += (long long)blockIdx.z * vs_in;  // vector blockIdx.z of a many-vector launch
    pin += (long long)blockIdx.z * vs_out;
    // workgroup x = group of the batch (item0 is a multiple of G); y = mode chunk
    const int g = item0 / G + xcd_block(blockIdx.x, gridDim.x);
    const int m = blockIdx.y * blockDim.x + threadIdx.x;
    if (m >= nm) return;
    Cx<R> ex{}, ey{}, ez{};
    if constexpr (sizeof(R) == 8) {
        const int b = m % n, a = (m / n) % h, c = m / (n * h);
        ex = ephase[c];
        ez = ephase[a];
        ey = ephase[b];
    }
    R sr[G], si[G];
#pragma unroll
    for (int t = 0; t < G; ++t) sr[t] = si[t] = R(0);
    for (int e = gptr[g]; e < gptr[g + 1]; ++e) {
        const unsigned long long st = gsten[e];  // uniform
        const Cx<R> av = pw_out[(size_t)(gslot[e] - slot0) * nm + m];
#pragma unroll
        for (int t = 0; t < G; ++t) {
            const int sten = (int)((st >> (8 * t)) & 255);
            if (sten == 255) continue;  // uniform
            R fr, fi;
            if constexpr (sizeof(R) == 8) {
                const int dz = sten / 9 - 1, dy = (sten / 3) % 3 - 1, dx = sten % 3 - 1;
                fr = 1;
                fi = 0;
                if (dz) {
                    fr = ez.re;
                    fi = dz > 0 ? ez.im : -ez.im;
                }
                if (dy) {
                    const R gi = dy > 0 ? ey.im : -ey.im, r = fr * ey.re - fi * gi;
                    fi = fma(fr, gi, fi * ey.re);
                    fr = r;
                }
                if (dx) {
                    const R gi = dx > 0 ? ex.im : -ex.im, r = fr * ex.re - fi * gi;
                    fi = fma(fr, gi, fi * ex.re);
                    fr = r;
                }
            } else {
                const Cx<R> f = shift0[(size_t)sten * nm + m];
                fr = f.re;
                fi = f.im;
            }
            sr[t] = fma(av.re, fr, fma(-av.im, fi, sr[t]));
            si[t] = fma(av.re, fi, fma(av.im, fr, si[t]));
        }
    }
    R rr = lscale;
    if constexpr (sizeof(R) == 8) rr = radial0[m] * lscale;
#pragma unroll
    for (int t = 0; t < G; ++t) {
        const int it = g * G + t - item0;  // item within the batch
        if (it < n_items) pin[(size_t)it * nm + m] = {sr[t] * rr, si[t] * rr};
    }
}

// down[c][b][a] (+)= 2 Re sum V(k1,a) V(k2,b) h(k3) V(k3,c) pin[k1][k3][k2], V = pw2poly
// (V(k, j) at V[k + n j]), h = 1/2 for k3 >= n/2 (planewave_to_proxy_potential).  One
// workgroup per (box, slice of a).
// The x step of whole boxes into HBM, for orders where the slices of k_pw2proxy would each
// re-read the box's incoming expansion (14 slices per box for FP64 at p = 28, 38 at p = 38):
// u1[it][a][k3][k2] = sum_k1 V(k1, a) pin[it][k1][k3][k2] for every a, one thread per column
// (k3, k2), the same sums as k_pw2proxy's x step.  k_pw2p_yz then takes each plane a of u1
// through the y and z steps.
template <class R, int P, int NPW>
__global__ __launch_bounds__(256) void k_pw2p_x(const Cx<R> *__restrict__ pin, const Cx<R> *__restrict__ V,
                                                int n_items, Cx<R> *__restrict__ u1) {
    chain_priority();
    constexpr int H = (NPW + 1) / 2, COL = H * NPW, PER = (COL + 255) / 256;  // workgroups per box
    const int lg = xcd_block(blockIdx.x, gridDim.x), it = lg / PER, col = (lg - it * PER) * 256 + (int)threadIdx.x;
    if (it >= n_items || col >= COL) return;
    const Cx<R> *X = pin + (size_t)it * NPW * COL;
    Cx<R> acc[P];
#pragma unroll
    for (int a = 0; a < P; ++a) acc[a] = {R(0), R(0)};
    for (int k1 = 0; k1 < NPW; ++k1) {
        const Cx<R> x = X[(size_t)k1 * COL + col];
#pragma unroll
        for (int a = 0; a < P; ++a) {
            if (a % 2 == 0) {
                const R m = V[k1 + NPW * a].re;
                acc[a].re = fma(m, x.re, acc[a].re);
                acc[a].im = fma(m, x.im, acc[a].im);
            } else {
                const R m = V[k1 + NPW * a].im;
                acc[a].re = fma(-m, x.im, acc[a].re);
                acc[a].im = fma(m, x.re, acc[a].im);
            }
        }
    }
    Cx<R> *out = u1 + (size_t)it * P * COL + col;
#pragma unroll
    for (int a = 0; a < P; ++a) out[(size_t)a * COL] = acc[a];
}

// Second pass of the two-pass plane-wave -> proxy transform (after k_pw2p_x), FP64 on the
// matrix cores: the y and z steps of one plane a per wavefront.  With G[k][j] the folded
// table (the non-zero part of V(k, j): real for even j, imaginary for odd j):
//   y:  R[k3][b] = sum_k2 u1.re[a][k3][k2] G[k2][b],  I[k3][b] = the same of u1.im;
//       U2[k3][b] = h(k3) (R, I) for even b, h(k3) (-I, R) for odd b
//   z:  Zr[c][b] = sum_k3 G[k3][c] U2.re[k3][b],  Zi[c][b] = the same of U2.im;
//       down[c][b][a] (+)= 2 Zr for even c, 2 (-Zi) for odd c
// (the parity of the output index picks the part, so each step forms both products and
// keeps one; a negated sum of fused multiply-adds is the sum of the negated terms, bit for
// bit).  y's output tile, lane l holding rows k3 = 4 q + l/16 of column b = l%16, is z's B
// operand for the 4-steps q of that tile, so U2 stays in registers.  LDS holds G transposed
// (Gt[k][j], zero-padded).  Every output sums its terms in the order of k_pw2proxy (k2, then
// k3 ascending).
template <int P, int NPW> struct Pw2pMfmaCfg {
    static constexpr int H = (NPW + 1) / 2;
    static constexpr int KS2 = (NPW + 3) / 4;     // y's 4-steps over k2
    static constexpr int MT = (H + 15) / 16;      // y's row tiles over k3
    static constexpr int KSZ = (H + 3) / 4;       // z's 4-steps over k3
    static constexpr int BT = (P + 15) / 16;      // column tiles over b, row tiles over c
    static constexpr int GR = 4 * (KS2 > 4 * MT ? KS2 : 4 * MT);  // rows of Gt
    static constexpr int LG = 16 * BT + 8;        // row stride of Gt (8 mod 16)
};

template <int P, int NPW>
__global__ __launch_bounds__(256) void k_pw2p_yz(const Cx<double> *__restrict__ u1, const double *__restrict__ F,
                                                 const int *__restrict__ box_down, const int *__restrict__ box_zero,
                                                 int item0, int n_items, double *__restrict__ down_base) {
    chain_priority();
    using Cfg = Pw2pMfmaCfg<P, NPW>;
    using M = Mfma16<double>;
    typedef M::acc_t acc_t;
    constexpr int H = Cfg::H, COL = H * NPW, PP = P * P, KS2 = Cfg::KS2, MT = Cfg::MT, KSZ = Cfg::KSZ, BT = Cfg::BT,
                  GR = Cfg::GR, LG = Cfg::LG, AG = (P + 3) / 4;  // 4 planes a per workgroup
    static_assert(NPW <= 64 && 16 * BT <= 64, "table rows of 64");
    __shared__ double Gt[GR * LG];  // Gt[k][j] = G[k][j] for k < n, j < p, else 0
    for (int i = threadIdx.x; i < GR * LG; i += 256) {
        const int k = i / LG, j = i - k * LG;
        Gt[i] = (k < NPW && j < P) ? F[j * 64 + k] : 0.0;
    }
    __syncthreads();
    const int lg = xcd_block(blockIdx.x, gridDim.x), it = lg / AG;
    const int a = (lg - it * AG) * 4 + __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    if (it >= n_items || a >= P) return;
    const int l = threadIdx.x & 63, kk = l >> 4, jj = l & 15;
    const Cx<double> *X = u1 + ((size_t)it * P + a) * COL;  // X[k3][k2]
    // y: R, I tiles (k3 tile mt, b tile nt)
    acc_t yr[MT][BT], yi[MT][BT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int nt = 0; nt < BT; ++nt) yr[mt][nt] = yi[mt][nt] = acc_t{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int ks = 0; ks < KS2; ++ks) {
        const int k2 = 4 * ks + kk;
        double g[BT];
#pragma unroll
        for (int nt = 0; nt < BT; ++nt) g[nt] = Gt[k2 * LG + 16 * nt + jj];  // B[k2][b]
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            const int k3 = 16 * mt + jj;
            Cx<double> x = {0.0, 0.0};
            if (k3 < H && k2 < NPW) x = X[k3 * NPW + k2];  // A[k3][k2]
#pragma unroll
            for (int nt = 0; nt < BT; ++nt) {
                yr[mt][nt] = M::mma(x.re, g[nt], yr[mt][nt]);
                yi[mt][nt] = M::mma(x.im, g[nt], yi[mt][nt]);
            }
        }
    }
    // U2 in place: element q of tile (mt, nt) is k3 = 16 mt + 4 q + kk, b = 16 nt + jj
    const bool bodd = jj & 1;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const double hw = (16 * mt + M::row(kk, q) >= NPW / 2) ? 0.5 : 1.0;
#pragma unroll
            for (int nt = 0; nt < BT; ++nt) {
                const double r = yr[mt][nt][q], i = yi[mt][nt][q];
                yr[mt][nt][q] = (bodd ? -i : r) * hw;
                yi[mt][nt][q] = (bodd ? r : i) * hw;
            }
        }
    // z: c tile ct, b tile nt; 4-step ks = 4 mt + q over k3
    double *down = down_base + (size_t)box_down[item0 + it] * P * PP;
    const bool zero = box_zero[item0 + it] != 0;
    const bool codd = kk & 1;  // parity of c = 16 ct + 4 q + kk
#pragma unroll
    for (int ct = 0; ct < BT; ++ct) {
        acc_t zr[BT], zi[BT];
#pragma unroll
        for (int nt = 0; nt < BT; ++nt) zr[nt] = zi[nt] = acc_t{0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                if (4 * mt + q < KSZ) {
                    const double gz = Gt[(16 * mt + 4 * q + kk) * LG + 16 * ct + jj];  // A[c][k3] = G[k3][c]
#pragma unroll
                    for (int nt = 0; nt < BT; ++nt) {
                        zr[nt] = M::mma(gz, yr[mt][nt][q], zr[nt]);
                        zi[nt] = M::mma(gz, yi[mt][nt][q], zi[nt]);
                    }
                }
            }
#pragma unroll
        for (int nt = 0; nt < BT; ++nt) {
            const int b = 16 * nt + jj;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int c = 16 * ct + M::row(kk, q);
                if (c < P && b < P) {
                    double *dst = down + ((size_t)c * P + b) * P + a;
                    const double v = codd ? -zi[nt][q] : zr[nt][q];
                    *dst = (zero ? 0.0 : *dst) + 2.0 * v;
                }
            }
        }
    }
}

template <class R, int P, int NPW, int BK = 0>
__global__ __launch_bounds__(256) void k_pw2proxy(const Cx<R> *__restrict__ pin, const Cx<R> *__restrict__ V,
                                                   const int *__restrict__ box_down, const int *__restrict__ box_zero,
                                                   int item0, int n_items, R *__restrict__ down_base,
                                                   long long vs_in = 0, long long vs_out = 0) {
    chain_priority();
    pin += (long long)blockIdx.z * vs_in;  // vector blockIdx.z of a many-vector launch
    down_base += (long long)blockIdx.z * vs_out;
    constexpr int H = (NPW + 1) / 2, COL = H * NPW, PP = P * P, half = NPW / 2, TS2 = OddStride<P>::v;
    constexpr int AC = Pw2pCfg<R, P, NPW, BK>::AC;
    __shared__ Cx<R> U1[AC * COL];       // [a][k3][k2]
    __shared__ Cx<R> U2[AC * H * TS2];   // [a][k3][b] rows of TS2
    // 1-D grid: (box, slice of a) at xcd_block index box * slices + slice
    constexpr int NS = Pw2pCfg<R, P, NPW, BK>::slices;
    const int lg = xcd_block(blockIdx.x, gridDim.x), it = lg / NS, slice = lg - it * NS;
    if (it >= n_items) return;
    const Cx<R> *X = pin + (size_t)it * NPW * COL;
    R *down = down_base + (size_t)box_down[item0 + it] * P * PP;
    const bool zero = box_zero[item0 + it] != 0;
    {
        const int a0 = slice * AC;
        const int na = min(AC, P - a0);
        // Each step's outputs are polynomial indices (a0 + a, b0 + b, c0 + c): the matrix row of
        // an output is real (even index) or imaginary (odd).  The parity of the first output
        // (uniform across a workgroup or a wavefront) selects a template instance, in which the
        // unrolled loops fold every output's parity.
        using Even = std::integral_constant<int, 0>;
        using Odd = std::integral_constant<int, 1>;
        // x: U1[a][k3][k2] = sum_k1 V(k1, a0 + a) pin[k1][k3][k2], column = (k3, k2)
        auto xstep = [&](auto par) {
            constexpr int A0P = decltype(par)::value;
            for (int col = threadIdx.x; col < COL; col += blockDim.x) {
                Cx<R> acc[AC];
#pragma unroll
                for (int a = 0; a < AC; ++a) acc[a] = {R(0), R(0)};
                for (int k1 = 0; k1 < NPW; ++k1) {
                    const Cx<R> x = X[(size_t)k1 * COL + col];
#pragma unroll
                    for (int a = 0; a < AC; ++a) {
                        if (a < na) {
                            if ((A0P + a) % 2 == 0) {
                                const R m = V[k1 + NPW * (a0 + a)].re;
                                acc[a].re = fma(m, x.re, acc[a].re);
                                acc[a].im = fma(m, x.im, acc[a].im);
                            } else {
                                const R m = V[k1 + NPW * (a0 + a)].im;
                                acc[a].re = fma(-m, x.im, acc[a].re);
                                acc[a].im = fma(m, x.re, acc[a].im);
                            }
                        }
                    }
                }
#pragma unroll
                for (int a = 0; a < AC; ++a)
                    if (a < na) U1[a * COL + col] = acc[a];
            }
        };
        if (a0 & 1) {
            xstep(Odd{});
        } else {
            xstep(Even{});
        }
        __syncthreads();
        // y: U2[a][k3][b] = h(k3) sum_k2 V(k2, b) U1[a][k3][k2]; slot = (column w = a H + k3,
        // segment of b, uniform across a wavefront)
        constexpr int SGY = Pw2pCfg<R, P, NPW, BK>::SGY, PSY = Pw2pCfg<R, P, NPW, BK>::PSY;
        const int ny = (na * H + 63) / 64 * 64 * SGY;
        for (int t = threadIdx.x; t < ny; t += blockDim.x) {
            int w, sg;
            t3_slot<SGY>(t, w, sg);
            if (w >= na * H) continue;
            const int k3 = w % H, b0 = sg * PSY;
            auto ystep = [&](auto par) {
                constexpr int B0P = decltype(par)::value;
                Cx<R> acc[PSY];
#pragma unroll
                for (int b = 0; b < PSY; ++b) acc[b] = {R(0), R(0)};
                for (int k2 = 0; k2 < NPW; ++k2) {
                    const Cx<R> x = U1[w * NPW + k2];
#pragma unroll
                    for (int b = 0; b < PSY; ++b) {
                        if (b0 + b < P) {
                            if ((B0P + b) % 2 == 0) {
                                const R m = V[k2 + NPW * (b0 + b)].re;
                                acc[b].re = fma(m, x.re, acc[b].re);
                                acc[b].im = fma(m, x.im, acc[b].im);
                            } else {
                                const R m = V[k2 + NPW * (b0 + b)].im;
                                acc[b].re = fma(-m, x.im, acc[b].re);
                                acc[b].im = fma(m, x.re, acc[b].im);
                            }
                        }
                    }
                }
                const R hw = (k3 >= half) ? R(0.5) : R(1);
#pragma unroll
                for (int b = 0; b < PSY; ++b)
                    if (b0 + b < P) U2[w * TS2 + b0 + b] = {acc[b].re * hw, acc[b].im * hw};
            };
            if (b0 & 1) ystep(Odd{});
            else ystep(Even{});
        }
        __syncthreads();
        // z: down[c][b][a0 + a] (+)= 2 Re sum_k3 V(k3, c) U2[a][k3][b]; slot = (column w = b na + a,
        // segment of c, uniform across a wavefront)
        constexpr int SGZ = Pw2pCfg<R, P, NPW, BK>::SGZ, PSZ = Pw2pCfg<R, P, NPW, BK>::PSZ;
        const int nz = (na * P + 63) / 64 * 64 * SGZ;
        for (int t = threadIdx.x; t < nz; t += blockDim.x) {
            int w, sg;
            t3_slot<SGZ>(t, w, sg);
            if (w >= na * P) continue;
            const int b = w / na, a = w - b * na, c0 = sg * PSZ;
            auto zstep = [&](auto par) {
                constexpr int C0P = decltype(par)::value;
                R acc[PSZ];
#pragma unroll
                for (int c = 0; c < PSZ; ++c) acc[c] = R(0);
                for (int k3 = 0; k3 < H; ++k3) {
                    const Cx<R> x = U2[(a * H + k3) * TS2 + b];
#pragma unroll
                    for (int c = 0; c < PSZ; ++c) {
                        if (c0 + c < P) {
                            if ((C0P + c) % 2 == 0) acc[c] = fma(V[k3 + NPW * (c0 + c)].re, x.re, acc[c]);
                            else acc[c] = fma(-V[k3 + NPW * (c0 + c)].im, x.im, acc[c]);
                        }
                    }
                }
                R *dst = down + (size_t)b * P + a0 + a;
#pragma unroll
                for (int c = 0; c < PSZ; ++c)
                    if (c0 + c < P)
                        dst[(size_t)(c0 + c) * PP] = (zero ? R(0) : dst[(size_t)(c0 + c) * PP]) + R(2) * acc[c];
            };
            if (c0 & 1) zstep(Odd{});
            else zstep(Even{});
        }
        __syncthreads();
    }
}

// pot_sorted[t] += sum C(a,b,c) T_a T_b T_c at the targets of one leaf per workgroup.  The
// coefficient planes C[c][.][.] are staged through LDS one at a time and read as broadcasts;
// each thread evaluates EV_TPT targets, T_a sits in registers and T_b, T_c follow the
// Chebyshev recurrence along their loops.
constexpr int EV_THREADS = 128, EV_TPT = 2;

template <class R, int P>
__global__ __launch_bounds__(EV_THREADS) void k_eval_targets(const R *__restrict__ down_base, const int *__restrict__ leaf_down,
                                                              const R *__restrict__ leaf_geom, const int *__restrict__ leaf_trg,
                                                              const P4<R> *__restrict__ trg, R *__restrict__ pot_sorted,
                                                              long long vs_in = 0, long long vs_out = 0) {
    chain_priority();
    down_base += (long long)blockIdx.z * vs_in;  // vector blockIdx.z of a many-vector launch
    pot_sorted += (long long)blockIdx.z * vs_out;
    constexpr int PP = P * P;
    __shared__ R plane[PP];
    const int lf = blockIdx.x;
    const R *C = down_base + (size_t)leaf_down[lf] * P * PP;
    const R cx = leaf_geom[4 * lf], cy = leaf_geom[4 * lf + 1], cz = leaf_geom[4 * lf + 2], sc = leaf_geom[4 * lf + 3];
    const int beg = leaf_trg[2 * lf], cnt = leaf_trg[2 * lf + 1];
    for (int t0 = 0; t0 < cnt; t0 += EV_THREADS * EV_TPT) {
        R tx[EV_TPT][P], y[EV_TPT], z[EV_TPT], s[EV_TPT], tcm1[EV_TPT], tc[EV_TPT];
#pragma unroll
        for (int i = 0; i < EV_TPT; ++i) {
            const int t = t0 + (int)threadIdx.x + EV_THREADS * i;
            const P4<R> pt = t < cnt ? trg[beg + t] : P4<R>{cx, cy, cz, R(0)};
            const R x = sc * (pt.x - cx);
            y[i] = sc * (pt.y - cy);
            z[i] = sc * (pt.z - cz);
            tx[i][0] = R(1);
            if (P > 1) tx[i][1] = x;
#pragma unroll
            for (int k = 2; k < P; ++k) tx[i][k] = R(2) * x * tx[i][k - 1] - tx[i][k - 2];
            s[i] = R(0);
            tcm1[i] = R(1);
            tc[i] = R(1);
        }
        for (int c = 0; c < P; ++c) {
            __syncthreads();
            for (int e = threadIdx.x; e < PP; e += EV_THREADS) plane[e] = C[(size_t)c * PP + e];
            __syncthreads();
#pragma unroll
            for (int i = 0; i < EV_TPT; ++i) {
                if (c == 1) {
                    tc[i] = z[i];
                } else if (c > 1) {
                    const R tn = R(2) * z[i] * tc[i] - tcm1[i];
                    tcm1[i] = tc[i];
                    tc[i] = tn;
                }
            }
            R sb[EV_TPT], tbm1[EV_TPT], tb[EV_TPT];
#pragma unroll
            for (int i = 0; i < EV_TPT; ++i) { sb[i] = R(0); tbm1[i] = R(1); tb[i] = R(1); }
            for (int b = 0; b < P; ++b) {
#pragma unroll
                for (int i = 0; i < EV_TPT; ++i) {
                    if (b == 1) {
                        tb[i] = y[i];
                    } else if (b > 1) {
                        const R tn = R(2) * y[i] * tb[i] - tbm1[i];
                        tbm1[i] = tb[i];
                        tb[i] = tn;
                    }
                }
                R sa[EV_TPT];
#pragma unroll
                for (int i = 0; i < EV_TPT; ++i) sa[i] = R(0);
#pragma unroll
                for (int a = 0; a < P; ++a) {
                    const R cv = plane[b * P + a];
#pragma unroll
                    for (int i = 0; i < EV_TPT; ++i) sa[i] = fma(cv, tx[i][a], sa[i]);
                }
#pragma unroll
                for (int i = 0; i < EV_TPT; ++i) sb[i] = fma(sa[i], tb[i], sb[i]);
            }
#pragma unroll
            for (int i = 0; i < EV_TPT; ++i) s[i] = fma(sb[i], tc[i], s[i]);
        }
#pragma unroll
        for (int i = 0; i < EV_TPT; ++i) {
            const int t = t0 + (int)threadIdx.x + EV_THREADS * i;
            if (t < cnt) pot_sorted[beg + t] += s[i];
        }
    }
}

// The same evaluation on the matrix cores, for p >= 18.  Per leaf and stage of targets
//   R[t, (c, b)] = sum_a T_a(x_t) C[(c, b), a]          (GEMM, a padded to 4s)
//   pot_t += sum_(c,b) R[t, (c, b)] T_b(y_t) T_c(z_t)
// with 16 x 16 x 4 products (Mfma16).  Wave w takes the (c, b) tiles w, w + NW, ..., whose B
// operands (the leaf's proxy rows) stay in registers for the whole leaf, so the proxy is read
// once per leaf, all its loads in flight together; the targets pass by in stages of TT tiles of
// 16.  Lane partials are reduced over each 16-lane row (halving the values with each exchange),
// then over the waves in a fixed order.  At p = 38 a wave's B operands would not fit its
// registers: the leaf's (c, b) tiles are taken in RH = 2 halves, each a pass over the leaf's
// targets that adds its part of the sum to the potentials.
// At p = 18 the vector kernel ran 18 dependent plane loads per leaf and took vector issue from
// the near field beside it.  Alone, FP32 / FP64: N = 1e3 48 / 69 -> 6 / 7 us, 3e4 88 / 131 ->
// 14 / 22, 2.5e5 164 / 332 -> 63 / 124, 1e6 256 / 492 -> 180 / 382.  What bounds it now: the
// matrix cores at about half their rate, then the stages' serial parts (tables, reduction).
template <int CTRL> __device__ __forceinline__ float row_dpp(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), CTRL, 0xF, 0xF, true));
}
template <int CTRL> __device__ __forceinline__ double row_dpp(double v) {
    const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
    const unsigned lo = __builtin_amdgcn_mov_dpp((int)(unsigned)u, CTRL, 0xF, 0xF, true);
    const unsigned hi = __builtin_amdgcn_mov_dpp((int)(unsigned)(u >> 32), CTRL, 0xF, 0xF, true);
    return __builtin_bit_cast(double, (unsigned long long)hi << 32 | lo);
}
// a = the lane's and its partner's a (upper lanes of each pair: b)
template <int CTRL, class R> __device__ __forceinline__ void row_fold(R &a, const R &b, int upper) {
    const R keep = upper ? +b : +a, give = upper ? +a : +b;
    a = keep + row_dpp<CTRL>(give);
}
template <class R, int P> struct EvMfmaCfg {
    static constexpr int RT = (P * P + 15) / 16;
    // (4 waves and more passes: two workgroups per CU, one's table building and reduction beside
    // the other's products; N = 1e6: 9 digits 1220 us with 7 waves in one pass, 1094 with 4 in
    // two; 12 digits 3781 us with 8 waves in two passes, 2994 with 4 in four)
    static constexpr int NW = 4;
    static constexpr int RH = P >= 38 ? 4 : (P >= 28 ? 2 : 1);  // passes over the leaf's targets
    static constexpr int MT = (RT + NW * RH - 1) / (NW * RH);  // (c, b) tiles per wave and pass
    static constexpr int TT = 2;                   // target tiles per stage
    static constexpr int NT = 16 * TT;             // targets per stage
    static constexpr int PA = (P + 3) / 4 * 4;
    // LDS row strides, in elements: odd, so that the 32 threads that write their targets' rows in
    // step and the 16 targets of an A read each fall on distinct banks (FP64 rows of 34 and 48:
    // 16-way conflicts of the writes, 23% of the kernel's LDS time at N = 1e6, 9 digits)
    static constexpr int LX = PA | 1, LY = P | 1;
    static_assert(P <= LY, "order above the table stride");
};
template <class R, int P>
__global__ __launch_bounds__((64 * EvMfmaCfg<R, P>::NW), 2) void k_eval_targets_mfma(
    const R *__restrict__ down_base, const int *__restrict__ leaf_down, const R *__restrict__ leaf_geom,
    const int *__restrict__ leaf_trg, const P4<R> *__restrict__ trg, R *__restrict__ pot_sorted, long long vs_in = 0,
    long long vs_out = 0) {
    chain_priority();
    using C = EvMfmaCfg<R, P>;
    using M = Mfma16<R>;
    constexpr int RT = C::RT, NW = C::NW, RH = C::RH, MT = C::MT, TT = C::TT, NT = C::NT, PA = C::PA, PP = P * P;
    static_assert(P <= PA, "order above the padded a count");
    static_assert(TT == 2, "the row reduction halves 8 values");
    constexpr int LX = C::LX, LY = C::LY;
    __shared__ R Tx[NT * LX], Ty[NT * LY], Tz[NT * LY], red[NW * NT];
    down_base += (long long)blockIdx.z * vs_in;  // vector blockIdx.z of a many-vector launch
    pot_sorted += (long long)blockIdx.z * vs_out;
    const int lf = blockIdx.x, lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int kk = lane >> 4, jj = lane & 15;
    const R *Cm = down_base + (size_t)leaf_down[lf] * P * PP;
    const R cx = leaf_geom[4 * lf], cy = leaf_geom[4 * lf + 1], cz = leaf_geom[4 * lf + 2], sc = leaf_geom[4 * lf + 3];
    const int beg = leaf_trg[2 * lf], cnt = leaf_trg[2 * lf + 1];
    for (int h = 0; h < RH; ++h) {
        // B operands of tile rt = w + NW (h MT + m): lane (kk, jj) supplies C[rt 16 + jj][4 ks + kk]
        R B[MT][PA / 4];
        int ob[MT], oc[MT];  // table offsets of its (c, b)
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            const int row = (w + NW * (h * MT + m)) * 16 + jj;
            oc[m] = row < PP ? row / P : 0;
            ob[m] = row < PP ? row % P : 0;
#pragma unroll
            for (int ks = 0; ks < PA / 4; ++ks) {
                const int a = 4 * ks + kk;
                B[m][ks] = (row < PP && a < P) ? Cm[(size_t)row * P + a] : R(0);
            }
        }
        for (int t0 = 0; t0 < cnt; t0 += NT) {
            __syncthreads();
            for (int task = threadIdx.x; task < 3 * NT; task += blockDim.x) {
                const int t = task % NT, d = task / NT;
                R *T = d == 0 ? Tx + t * LX : (d == 1 ? Ty + t * LY : Tz + t * LY);
                const int len = d == 0 ? PA : P;
                if (t0 + t < cnt) {
                    const P4<R> pt = trg[beg + t0 + t];
                    const R x = sc * (d == 0 ? pt.x - cx : (d == 1 ? pt.y - cy : pt.z - cz));
                    R ta = R(1), tb = x;
                    T[0] = R(1);
                    T[1] = x;
                    for (int k = 2; k < P; ++k) {
                        const R tn = R(2) * x * tb - ta;
                        T[k] = tn;
                        ta = tb;
                        tb = tn;
                    }
                    for (int k = P; k < len; ++k) T[k] = R(0);
                } else {
                    for (int k = 0; k < len; ++k) T[k] = R(0);
                }
            }
            __syncthreads();
            R A[TT][PA / 4];
#pragma unroll
            for (int tt = 0; tt < TT; ++tt)
#pragma unroll
                for (int ks = 0; ks < PA / 4; ++ks) A[tt][ks] = Tx[(tt * 16 + jj) * LX + 4 * ks + kk];
            R part[4 * TT];
#pragma unroll
            for (int e = 0; e < 4 * TT; ++e) part[e] = R(0);
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                const int rt = w + NW * (h * MT + m);
                if (rt >= RT) break;  // wave-uniform
                typename M::acc_t D[TT];
#pragma unroll
                for (int tt = 0; tt < TT; ++tt) D[tt] = typename M::acc_t{R(0), R(0), R(0), R(0)};
#pragma unroll
                for (int ks = 0; ks < PA / 4; ++ks)
#pragma unroll
                    for (int tt = 0; tt < TT; ++tt) D[tt] = M::mma(A[tt][ks], B[m][ks], D[tt]);
                // D[tt][e] = R[target tt 16 + M::row(kk, e), (c, b) = rt 16 + jj]
#pragma unroll
                for (int tt = 0; tt < TT; ++tt)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const int t = tt * 16 + M::row(kk, e);
                        part[4 * tt + e] =
                            fma(D[tt][e], Ty[t * LY + ob[m]] * Tz[t * LY + oc[m]], part[4 * tt + e]);
                    }
            }
            // sum over the 16 lanes of each row (the (c, b) columns): 8 values per lane, halved with
            // each of three exchanges (partners i ^ 15, i ^ 7, i ^ 3, then i ^ 1: DPP moves); lane
            // jj ends with value 4 tt + e = jj / 2.  (Unary pluses: a conditional between array
            // elements would select their addresses.)
            row_fold<0x140>(part[0], part[4], jj & 8);
            row_fold<0x140>(part[1], part[5], jj & 8);
            row_fold<0x140>(part[2], part[6], jj & 8);
            row_fold<0x140>(part[3], part[7], jj & 8);
            row_fold<0x141>(part[0], part[2], jj & 4);
            row_fold<0x141>(part[1], part[3], jj & 4);
            row_fold<0x1B>(part[0], part[1], jj & 2);
            part[0] += row_dpp<0xB1>(part[0]);
            if ((jj & 1) == 0) red[w * NT + (jj >> 3) * 16 + M::row(kk, (jj >> 1) & 3)] = part[0];
            __syncthreads();
            for (int t = threadIdx.x; t < NT; t += blockDim.x) {
                if (t0 + t < cnt) {
                    R v = R(0);
#pragma unroll
                    for (int q = 0; q < NW; ++q) v += red[q * NT + t];
                    pot_sorted[beg + t0 + t] += v;
                }
            }
        }
    }
}

// ------------------------------------------------------------------ near field
// Residual u = P((r - bs/2) 2/bs) / r for 1e-30 < r^2 < bs^2, summed over the list1
// sources of every target.  For fewer than 6 digits P is applied in r^2 with an even/odd
// split (monomial coefficients per bs, prepared on the host), as laplace_3d_poly_all_pairs
// does.
//
// Work item = one wavefront = up to 64 targets of one leaf (consecutive in the leaf's
// Morton order, so the item is spatially compact).  The geometry is fixed for the life of a
// tree, so which sources can reach which wavefront is decided once, at construction
// (k_near_steps): a step is one source of one list1 entry for which at least one lane of
// the wavefront is in support.  The evaluation walks only the steps, in the order the
// construction found them, and applies the per-lane support test to each; sources are read
// with wave-uniform addresses.
//
// Coordinates are relative to each point's leaf centre; geom[e] = (centre of the target
// leaf - centre of the source leaf, bs), so r = |(t + off) - s|.  Each list entry is
// summed in R and the per-target total in FP64.
constexpr int NF_CHUNK = 4;
constexpr int NF_SPLIT_STRIDE = 16;  // coefficient stride of the even/odd table
// steps whose sources are loaded together (scalar loads: U points in SGPRs); the step list
// is padded by NF_STEP_PAD valid indices so a group may read past the end of its run
template <class R> constexpr int nf_unroll() { return sizeof(R) == 4 ? 8 : 4; }
constexpr int NF_STEP_PAD = 16;

struct NfEntry { int sbeg, scnt, cbase, cfidx; };

// Step lists, once per tree.  Sources of every leaf are cut into chunks of NF_CHUNK
// consecutive (Morton-ordered) points with bounding boxes cbox; for each list1 entry the 64
// lanes test 64 chunks at once against the item's box wbox (shifted into the source leaf's
// frame), evaluated with the same rounded operations as the per-pair r^2 so that it never
// drops a pair the per-pair test keeps; the sources of kept chunks are then tested per lane.
// PASS 0 writes the step count of the k-th entry of item i to cnt[ie_base[i] + k] and adds
// the in-support pairs to *pairs; PASS 1 writes the steps' source indices from
// ie_ptr[ie_base[i] + k] on.
template <class R, int PASS>
__global__ __launch_bounds__(256) void k_near_steps(const P4<R> *__restrict__ src, const P4<R> *__restrict__ trg,
                                                     const int4 *__restrict__ items, const P4<R> *__restrict__ wbox,
                                                     const int *__restrict__ l1_ptr, const NfEntry *__restrict__ l1,
                                                     const P4<R> *__restrict__ geom, const P4<R> *__restrict__ cbox,
                                                     const int *__restrict__ ie_base, int *__restrict__ cnt,
                                                     const long long *__restrict__ ie_ptr, int *__restrict__ step_src,
                                                     unsigned long long *__restrict__ pairs, int n_items) {
    const int item = blockIdx.x * (blockDim.x >> 6) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (item >= n_items) return;  // whole wavefront
    const int lane = threadIdx.x & 63;
    const int4 it = items[item];
    const bool active = lane < it.y;
    const P4<R> me = active ? trg[it.x + lane] : P4<R>{R(1e18), R(1e18), R(1e18), R(0)};
    const P4<R> blo = wbox[2 * item], bhi = wbox[2 * item + 1];
    const int eb = l1_ptr[it.z], base = ie_base[item];
    unsigned long long np = 0;
    for (int e = eb; e < l1_ptr[it.z + 1]; ++e) {
        const NfEntry E = l1[e];
        const P4<R> gm = geom[e];
        const R bs = gm.w, d2max = bs * bs;
        const R tx = me.x + gm.x, ty = me.y + gm.y, tz = me.z + gm.z;
        const R lx = blo.x + gm.x, ly = blo.y + gm.y, lz = blo.z + gm.z;
        const R hx = bhi.x + gm.x, hy = bhi.y + gm.y, hz = bhi.z + gm.z;
        const int nch = (E.scnt + NF_CHUNK - 1) / NF_CHUNK;
        long long out = PASS == 1 ? ie_ptr[base + e - eb] : 0;
        int steps = 0;
        for (int c0 = 0; c0 < nch; c0 += 64) {
            bool keep = false;
            if (c0 + lane < nch) {
                const P4<R> cl = cbox[2 * (E.cbase + c0 + lane)], ch = cbox[2 * (E.cbase + c0 + lane) + 1];
                const R dx = fmax(fmax(cl.x - hx, lx - ch.x), R(0));
                const R dy = fmax(fmax(cl.y - hy, ly - ch.y), R(0));
                const R dz = fmax(fmax(cl.z - hz, lz - ch.z), R(0));
                keep = fma(dx, dx, fma(dy, dy, dz * dz)) < d2max;
            }
            unsigned long long mask = __ballot(keep);
            while (mask) {
                const int k = __ffsll((unsigned long long)mask) - 1;
                mask &= mask - 1;
                const int s0 = E.sbeg + (c0 + k) * NF_CHUNK;
                const int ns = min(NF_CHUNK, E.sbeg + E.scnt - s0);
                for (int j = 0; j < ns; ++j) {
                    const P4<R> q = src[s0 + j];
                    const R dx = tx - q.x, dy = ty - q.y, dz = tz - q.z;
                    const R r2 = fma(dx, dx, fma(dy, dy, dz * dz));
                    const unsigned long long in = __ballot(r2 < d2max && r2 > R(1e-30));
                    if (in) {
                        if (PASS == 1 && lane == 0) step_src[out] = s0 + j;
                        out += 1;
                        steps += 1;
                        np += __popcll(in);
                    }
                }
            }
        }
        if (PASS == 0 && lane == 0) cnt[base + e - eb] = steps;
    }
    if (PASS == 0 && lane == 0) atomicAdd(pairs, np);
}

// Residual evaluation over the step lists (steps of the k-th entry of item i:
// step_src[ie_ptr[ie_base[i] + k] .. ie_ptr[ie_base[i] + k + 1])).
template <class R, int NC, bool SPLIT>
__global__ __launch_bounds__(1024) void k_near_field(const P4<R> *__restrict__ src, const P4<R> *__restrict__ trg,
                                                     const int4 *__restrict__ items, const int *__restrict__ l1_ptr,
                                                     const NfEntry *__restrict__ l1, const P4<R> *__restrict__ geom,
                                                     const int *__restrict__ ie_base, const long long *__restrict__ ie_ptr,
                                                     const int *__restrict__ step_src, const R *__restrict__ coeffs,
                                                     R *__restrict__ pot_sorted, int item0, int item1, long long vs_src = 0,
                                                     long long vs_pot = 0) {
    src += (long long)blockIdx.z * vs_src;  // component blockIdx.z of a quasi-periodic pass
    pot_sorted += (long long)blockIdx.z * vs_pot;
    // wave index made wave-uniform explicitly, so everything derived from it lives in SGPRs
    const int item = item0 + xcd_block(blockIdx.x, gridDim.x) * (blockDim.x >> 6) +
                     __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (item >= item1) return;  // whole wavefront
    const int lane = threadIdx.x & 63;
    const int4 it = items[item];  // (first target, count, target-leaf list index, -)
    const bool active = lane < it.y;
    const P4<R> me = active ? trg[it.x + lane] : P4<R>{R(1e18), R(1e18), R(1e18), R(0)};
    R c[NC];
    if (!SPLIT) {
#pragma unroll
        for (int i = 0; i < NC; ++i) c[i] = coeffs[i];
    }
    // FP64: leading coefficient in a VGPR, so each Horner FMA reads at most one SGPR (no copy
    // per step), and the charge product inside the support branch.  Measured at N=1e6: the
    // FP64 near field 3.60 -> 3.43 ms and evaluate() 4.82 -> 4.67 ms at 6 digits; in FP32 the
    // same change slows evaluate() (3.02 -> 3.10 ms) although the kernel alone gains 1%.
    constexpr bool trim = sizeof(R) == 8;
    const R ctop = SPLIT ? R(0) : (trim ? c[NC - 1] + (R)vgpr_zero() : c[NC - 1]);
    const int eb = l1_ptr[it.z];
    const long long *iep = ie_ptr + ie_base[item] - eb;
    double acc = 0;
    for (int e = eb; e < l1_ptr[it.z + 1]; ++e) {
        const long long sb = iep[e], se = iep[e + 1];
        if (sb == se) continue;
        const P4<R> gm = geom[e];
        const R bs = gm.w, d2max = bs * bs, rsc = R(2) / bs, cen = -bs / R(2);
        const R tx = me.x + gm.x, ty = me.y + gm.y, tz = me.z + gm.z;
        if (SPLIT) {
            const int cf = l1[e].cfidx;
#pragma unroll
            for (int i = 0; i < NC; ++i) c[i] = coeffs[cf * NF_SPLIT_STRIDE + i];
        }
        constexpr int U = nf_unroll<R>();
        const int *sp = step_src + sb;
        const int cnt = (int)(se - sb);
        R ea = 0;
        for (int g = 0; g < cnt; g += U) {
            // all U indices and then all U points are requested before the first use
            int id[U];
#pragma unroll
            for (int j = 0; j < U; ++j) id[j] = sp[g + j];
            P4<R> qs[U];
#pragma unroll
            for (int j = 0; j < U; ++j) qs[j] = src[id[j]];
            // distances of all U points first and every point used unconditionally, so that
            // all point loads are in flight before the first wait; steps past the run get
            // r^2 = bs^2, outside the support
            R r2s[U];
#pragma unroll
            for (int j = 0; j < U; ++j) {
                const R dx = tx - qs[j].x, dy = ty - qs[j].y, dz = tz - qs[j].z;
                const R r2 = fma(dx, dx, fma(dy, dy, dz * dz));
                r2s[j] = g + j < cnt ? r2 : d2max;
            }
            // (empty statements that keep the U distances and charges ahead of the first step:
            // the compiler would otherwise sink them, and with them the point loads, into
            // later steps)
#pragma unroll
            for (int j = 0; j < U; ++j) {
                if (trim) asm volatile("" ::"v"(r2s[j]), "s"(qs[j].w));
                else asm volatile("" ::"v"(r2s[j]));
            }
#pragma unroll
            for (int j = 0; j < U; ++j) {
                const R r2 = r2s[j];
                R u = 0;
                if (r2 < d2max && r2 > R(1e-30)) {
                    const R rinv = rsqrt_full<R>(r2);
                    if (SPLIT) {
                        constexpr int SE = (NC - 1) & ~1, SO = ((NC - 2) & ~1) + 1;
                        R Ev = c[SE];
#pragma unroll
                        for (int i = SE - 2; i >= 0; i -= 2) Ev = fma(Ev, r2, c[i]);
                        R Od = c[SO];
#pragma unroll
                        for (int i = SO - 2; i >= 0; i -= 2) Od = fma(Od, r2, c[i]);
                        u = fma(Ev, rinv, Od);
                    } else {
                        const R x = fma(r2, rinv, cen) * rsc;
                        R p = ctop;
#pragma unroll
                        for (int i = NC - 2; i >= 0; --i) p = fma(p, x, c[i]);
                        u = p * rinv;
                    }
                    if (trim) ea = fma(u, qs[j].w, ea);
                }
                if (!trim) ea = fma(u, qs[j].w, ea);
            }
        }
        acc += (double)ea;
    }
    if (active) pot_sorted[it.x + lane] += (R)acc;
}

// ---------------------------------------------------------- near field in quad rows (FP32)
// The wavefront's 64 targets form 16 rows of 4 (lane l = 4 g + j: row g, target it.x + l).
// Every row walks a step list of its own: the sources (over all list1 entries of the target
// leaf, in entry order, and in walk order inside an entry) that reach at least one of its 4
// targets.  The 4 targets of a row are much closer together than the 64 of the wavefront, so
// fewer of a step's lanes fall outside the support: at N=1e6 (uniform) about 54% of the lanes
// of a step are in support against 34% when the whole wavefront shares one list.
//
// Step lists (built once per tree, k_near_rows_build): per item, K steps per row (K = the
// longest row's count rounded up to 4; shorter rows are padded with a far sentinel point),
// stored as source indices in blocks of 4 steps: block b holds at element 4 g + j the source
// of step 4 b + j of row g, so lane l loads element l of each block (one coalesced 256-byte
// read) and the 4 points of a row's block reach the row's lanes by DPP quad broadcasts.
// Per (item, row) the non-empty entries are listed as slots (entry ordinal, end step), ending
// with a terminator slot (nothing in support).
//
// For each target the in-support sources appear in its row's list in the same order as in
// the wavefront's list of k_near_field, each entry's sum is formed the same way and added to
// the FP64 total in entry order (entries without steps add nothing, there as 0.0 here), so
// the potentials equal k_near_field's bit for bit.
constexpr int NF_ROWS = 16;          // rows of 4 targets per wavefront
constexpr int NF_ROW_PAD = 2 * 64;   // sentinel indices past the last block (loads run one block ahead)
// Bit 31 of a step index flags a row's entry switch at that step (the first step of each of
// the row's entries but its first).  Readers form byte offsets as (unsigned)index * size in
// 32 bits, which drops the flag (source indices stay below 2^26).
constexpr int NF_STEP_ENTRY = (int)0x80000000u;

template <int S>
__device__ __forceinline__ float quad_bcast(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), S * 0x55, 0xF, 0xF, true));
}

// ea += q(lane 4 g + S) * u in one DPP-broadcast FMA (the same fused multiply-add as
// fmaf(quad_bcast<S>(q), u, ea)), led by s_nop 1: the two wait states a DPP read needs after a
// VALU write of its source (the compiler does not check hazards inside inline asm).
#define PDMK_FMAC_QUAD1(SEL) \
    asm("s_nop 1\n"          \
        "v_fmac_f32_dpp %0, %1, %2 quad_perm:[" SEL "] row_mask:0xf bank_mask:0xf bound_ctrl:1" : "+v"(ea) : "v"(q), "v"(u))
template <int S>
__device__ __forceinline__ void fmac_quad1(float &ea, float q, float u) {
    if constexpr (S == 0) PDMK_FMAC_QUAD1("0,0,0,0");
    if constexpr (S == 1) PDMK_FMAC_QUAD1("1,1,1,1");
    if constexpr (S == 2) PDMK_FMAC_QUAD1("2,2,2,2");
    if constexpr (S == 3) PDMK_FMAC_QUAD1("3,3,3,3");
}
#undef PDMK_FMAC_QUAD1

// *(T *)((char *)base + off) with a 32-bit unsigned byte offset: a wave-uniform base and a
// per-lane offset that the address computation needs no 64-bit arithmetic for
template <class T, class B>
__device__ __forceinline__ T nf_load_u32(const B *base, unsigned off) {
    return *reinterpret_cast<const T *>(reinterpret_cast<const char *>(base) + off);
}

// PASS 0: steps of row g in the k-th entry of item i -> cnt[(ie_base[i] + k) * 16 + g], and the
// in-support pairs added to *pairs.  PASS 1: the source indices into the row blocks from
// steps + wave_base[i] (the item's K, as built on the host, in items[i].w).  With parts
// (PASS 1) items come in n_parts parts each: wavefront p of item i writes the lists of entries
// parts[p' ].x .. parts[p'].y - 1, p' = i n_parts + p, from wave_base[p'].
template <class R, int PASS>
__global__ __launch_bounds__(256) void k_near_rows_build(
    const P4<R> *__restrict__ src, const P4<R> *__restrict__ trg, const int4 *__restrict__ items,
    const P4<R> *__restrict__ wbox, const int *__restrict__ l1_ptr, const NfEntry *__restrict__ l1,
    const P4<R> *__restrict__ geom, const P4<R> *__restrict__ cbox, const int *__restrict__ ie_base,
    int *__restrict__ cnt, const long long *__restrict__ wave_base, int *__restrict__ steps,
    unsigned long long *__restrict__ pairs, int n_items, const int2 *__restrict__ parts = nullptr, int n_parts = 1) {
    const int wave = blockIdx.x * (blockDim.x >> 6) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (wave >= n_items * n_parts) return;  // whole wavefront
    const int item = wave / n_parts;
    const int lane = threadIdx.x & 63;
    const int4 it = items[item];
    const bool active = lane < it.y;
    const P4<R> me = active ? trg[it.x + lane] : P4<R>{R(1e18), R(1e18), R(1e18), R(0)};
    const P4<R> blo = wbox[2 * item], bhi = wbox[2 * item + 1];
    const int eb = l1_ptr[it.z], base = ie_base[item];
    int *out = PASS == 1 ? steps + wave_base[wave] + lane : nullptr;
    unsigned long long np = 0;
    int k_row = 0;  // steps of this lane's row so far (the same in the row's 4 lanes)
    const int e_first = parts ? eb + parts[wave].x : eb, e_last = parts ? eb + parts[wave].y : l1_ptr[it.z + 1];
    for (int e = e_first; e < e_last; ++e) {
        const NfEntry E = l1[e];
        const P4<R> gm = geom[e];
        const R bs = gm.w, d2max = bs * bs;
        const R tx = me.x + gm.x, ty = me.y + gm.y, tz = me.z + gm.z;
        const R lx = blo.x + gm.x, ly = blo.y + gm.y, lz = blo.z + gm.z;
        const R hx = bhi.x + gm.x, hy = bhi.y + gm.y, hz = bhi.z + gm.z;
        const int nch = (E.scnt + NF_CHUNK - 1) / NF_CHUNK;
        int c_row = 0;
        for (int c0 = 0; c0 < nch; c0 += 64) {
            bool keep = false;
            if (c0 + lane < nch) {
                const P4<R> cl = cbox[2 * (E.cbase + c0 + lane)], ch = cbox[2 * (E.cbase + c0 + lane) + 1];
                const R dx = fmax(fmax(cl.x - hx, lx - ch.x), R(0));
                const R dy = fmax(fmax(cl.y - hy, ly - ch.y), R(0));
                const R dz = fmax(fmax(cl.z - hz, lz - ch.z), R(0));
                keep = fma(dx, dx, fma(dy, dy, dz * dz)) < d2max;
            }
            unsigned long long mask = __ballot(keep);
            while (mask) {
                const int k = __ffsll((unsigned long long)mask) - 1;
                mask &= mask - 1;
                const int s0 = E.sbeg + (c0 + k) * NF_CHUNK;
                const int ns = min(NF_CHUNK, E.sbeg + E.scnt - s0);
                for (int j = 0; j < ns; ++j) {
                    const P4<R> q = src[s0 + j];
                    const R dx = tx - q.x, dy = ty - q.y, dz = tz - q.z;
                    const R r2 = fma(dx, dx, fma(dy, dy, dz * dz));
                    const unsigned long long in = __ballot(r2 < d2max && r2 > R(1e-30));
                    np += __popcll(in);
                    if ((in >> (lane & ~3)) & 0xFull) {
                        // bit 31: the row's step starts an entry after its first
                        if (PASS == 1 && (k_row & 3) == (lane & 3))
                            out[(size_t)(k_row >> 2) * 64] = (s0 + j) | (c_row == 0 && k_row > 0 ? NF_STEP_ENTRY : 0);
                        ++k_row;
                        ++c_row;
                    }
                }
            }
        }
        if (PASS == 0 && (lane & 3) == 0) cnt[(size_t)(base + e - eb) * NF_ROWS + (lane >> 2)] = c_row;
    }
    if (PASS == 0 && lane == 0) atomicAdd(pairs, np);
}

// float4 of a list entry's geometry in k_near_rows' LDS
template <int NC, bool SPLIT> __host__ __device__ constexpr int nf_geo_f4() { return SPLIT ? 1 + (NC + 3) / 4 : 2; }

// Residual evaluation over the row step lists (FP32, NC coefficients in the x form).  Row g
// of item i lists its non-empty entries in slots rslot[(rs_base[i] + s) * 16 + g] =
// (end step << 8) | ordinal of the entry in the target leaf's list1, followed by a terminator
// (ordinal = number of entries: bs = 0, nothing in support).  Each wavefront copies its leaf's
// entry geometry (offset, bs, 2/bs, -bs/2, bs^2) and its rows' slots into LDS (ne_max + 1
// entries per wavefront), so an entry switch reads LDS only.  In LDS a slot is decoded ahead:
// (end step << 16) | byte offset of the entry's geometry from the LDS base (end steps below
// 2^16, and the workgroup's LDS below 64 KiB, both checked on the host; the terminator's end
// is clamped to 2^16 - 1, past every step).
// S > 1: trees with few items (N = 1e4: 192 wavefronts for 1024 SIMDs, each a serial walk of
// 1300 steps, 174 us).  A workgroup of S waves takes one item, each wave the row lists of its
// share of the list1 entries (items[item S + wave]); the entries' sums meet in LDS and are
// added in entry order, so the potentials are those of S = 1 bit for bit (73 us with S = 8;
// near_parts() has the other sizes).
// V = 2 (quasi-periodic): the residual formed once for two charges, the second from the copy of
// the sources vs_src further on (potentials vs_pot further on); each component's sums are those
// of V = 1.  (N = 1e5, beside the chain: 404 us against 504 for the two components along z.)
// SPLIT (fewer than 6 digits): the residual as two polynomials in r^2 (k_near_field), whose
// coefficients depend on the entry's bs: a row reads its entry's NC coefficients with the entry's
// geometry.  N = 4e5, 3 digits: 500 us alone with one list per wavefront, 300 with row lists.
template <int NC, int S, int V, bool SPLIT>
__global__ __launch_bounds__(1024) void k_near_rows(const P4<float> *__restrict__ src, const P4<float> *__restrict__ trg,
                                                   const int4 *__restrict__ items, const int *__restrict__ l1_ptr,
                                                   const P4<float> *__restrict__ geom, const int *__restrict__ rs_base,
                                                   const int *__restrict__ rslot, const long long *__restrict__ wave_base,
                                                   const int *__restrict__ steps, const float *__restrict__ coeffs,
                                                   float *__restrict__ pot_sorted, int item0, int item1, int ne_max,
                                                   long long vs_src = 0, long long vs_pot = 0,
                                                   const NfEntry *__restrict__ l1 = nullptr) {
    extern __shared__ float4 nf_lds[];
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int item = S > 1 ? (item0 + (int)blockIdx.x) * S + w
                           : item0 + xcd_block(blockIdx.x, gridDim.x) * (blockDim.x >> 6) + w;
    if (S == 1 && item >= item1) return;  // whole wavefront (no workgroup barrier below)
    const int lane = threadIdx.x & 63, g = lane >> 2;
    const int4 it = items[item];  // (first target, count, target-leaf list index, K)
    // this wavefront's LDS: ne_max + 1 entries x GS float4 (offset, bs^2, then 2/bs and -bs/2, or the
    // coefficients), then (ne_max + 1) x 16 slots
    constexpr int GS = nf_geo_f4<NC, SPLIT>();
    float4 *geo = nf_lds + (size_t)w * (ne_max + 1) * (GS + 4);
    int *slots = reinterpret_cast<int *>(geo + GS * (ne_max + 1));
    const int eb = l1_ptr[it.z], ne = l1_ptr[it.z + 1] - eb;
    // S > 1: the entries' sums [V][ne + 1][64]
    float *sums = reinterpret_cast<float *>(nf_lds + (size_t)S * (ne_max + 1) * (GS + 4));
    if (S > 1) {
        for (int k = threadIdx.x; k < V * (ne + 1) * 64; k += 64 * S) sums[k] = 0;
        __syncthreads();
    }
    for (int e = lane; e <= ne; e += 64) {
        const P4<float> gm = e < ne ? geom[eb + e] : P4<float>{0.0f, 0.0f, 0.0f, 0.0f};
        const float bs = gm.w;
        geo[GS * e] = make_float4(gm.x, gm.y, gm.z, bs * bs);
        if constexpr (SPLIT) {
            const float *ce = coeffs + (e < ne ? l1[eb + e].cfidx : 0) * NF_SPLIT_STRIDE;
            float *o = reinterpret_cast<float *>(geo + GS * e + 1);
#pragma unroll
            for (int i = 0; i < 4 * (GS - 1); ++i) o[i] = i < NC ? ce[i] : 0.0f;
        } else {
            geo[GS * e + 1] = make_float4(e < ne ? 2.0f / bs : 0.0f, -bs / 2.0f, 0.0f, 0.0f);
        }
    }
    const int *rs = rslot + (size_t)rs_base[item] * NF_ROWS;
    const int n_slots = S > 1 ? rs_base[item + 1] - rs_base[item] : ne + 1;
    const unsigned geo_off = (unsigned)((const char *)geo - (const char *)nf_lds);
    for (int k = lane; k < n_slots * NF_ROWS; k += 64) {
        const int v = rs[k];
        slots[k] = (int)(((unsigned)min(v >> 8, 0xffff) << 16) | (geo_off + 16u * GS * (unsigned)(v & 255)));
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const bool active = lane < it.y;
    const P4<float> me = active ? trg[it.x + lane] : P4<float>{1e18f, 1e18f, 1e18f, 0.0f};
    float c[NC];
#pragma unroll
    for (int i = 0; i < NC; ++i) c[i] = SPLIT ? 0.0f : coeffs[i];
    // the second-highest coefficient in a vector register: the first Horner step then takes
    // the highest from a scalar register and needs no copy per pair (one scalar operand per
    // FMA)
    float c_next = 0;
    if constexpr (!SPLIT) asm("v_mov_b32 %0, %1" : "=v"(c_next) : "s"(c[NC - 2]));
    float tx = 0, ty = 0, tz = 0, d2max = 0, rsc = 0, cen = 0;
    int end = 0;
    const int *slot = slots + g;  // the row's next slot
    double acc[V];
    float ea[V];
#pragma unroll
    for (int v = 0; v < V; ++v) {
        acc[v] = 0;
        ea[v] = 0;
    }
    float *sum = sums + (size_t)ne * 64 + lane;  // the current entry's (row ne: none)
    auto enter = [&]() {  // the row's next non-empty entry (or the terminator)
#pragma unroll
        for (int v = 0; v < V; ++v) {
            if (S > 1) sum[v * (ne + 1) * 64] = ea[v];
            else acc[v] += (double)ea[v];
            ea[v] = 0;
        }
        const unsigned v = (unsigned)*slot;
        slot += NF_ROWS;
        end = (int)(v >> 16);
        if (S > 1) sum = sums + ((v & 0xffffu) - geo_off) / (16u * GS) * 64u + lane;
        const float4 *ge = reinterpret_cast<const float4 *>(reinterpret_cast<const char *>(nf_lds) + (v & 0xffffu));
        const float4 a = ge[0], b = ge[1];
        tx = me.x + a.x;
        ty = me.y + a.y;
        tz = me.z + a.z;
        d2max = a.w;
        if constexpr (SPLIT) {
            const float *ce = reinterpret_cast<const float *>(ge + 1);
#pragma unroll
            for (int i = 0; i < NC; ++i) c[i] = ce[i];
        } else {
            rsc = b.x;
            cen = b.y;
        }
    };
    enter();
    const int K = it.w;
    // step indices: block b at sb + 64 b, element `lane`; the loads below take a wave-uniform
    // base and a 32-bit lane offset (one address instruction per load)
    const int *sb = steps + wave_base[item];
    auto index = [&](int b) { return nf_load_u32<int>(sb + (size_t)b * 64, (unsigned)lane * 4u); };
    auto point = [&](int id) { return nf_load_u32<P4<float>>(src, (unsigned)id * 16u); };
    const P4<float> *src1 = src + vs_src;
    auto charge1 = [&](int id) { return V > 1 ? nf_load_u32<float>(&src1->w, (unsigned)id * 16u) : 0.0f; };
    // m: ballot of the block's entry flags, bit 4 g + s = row g switches entries at step s
    auto block = [&](const P4<float> &pc, float q1, unsigned long long m, int k) {
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            // rows reach their entries' ends at different steps; the wave-wide test is scalar
            // (the empty asm keeps the compiler from folding the per-lane test into it, which
            // would issue that test at every step)
            if ((m >> s) & 0x1111111111111111ull) {
                asm volatile("");
                if (k + s >= end) enter();
            }
            float px, py, pz;
            switch (s) {
            case 0: px = quad_bcast<0>(pc.x); py = quad_bcast<0>(pc.y); pz = quad_bcast<0>(pc.z); break;
            case 1: px = quad_bcast<1>(pc.x); py = quad_bcast<1>(pc.y); pz = quad_bcast<1>(pc.z); break;
            case 2: px = quad_bcast<2>(pc.x); py = quad_bcast<2>(pc.y); pz = quad_bcast<2>(pc.z); break;
            default: px = quad_bcast<3>(pc.x); py = quad_bcast<3>(pc.y); pz = quad_bcast<3>(pc.z); break;
            }
            // (source - target: the negated difference, exactly, so r^2 is the same)
            const float dx = px - tx, dy = py - ty, dz = pz - tz;
            const float r2 = fmaf(dx, dx, fmaf(dy, dy, dz * dz));
            float u = 0;
            if (r2 < d2max && r2 > 1e-30f) {
                const float rinv = rsqrt_full<float>(r2);
                if constexpr (SPLIT) {
                    constexpr int SE = (NC - 1) & ~1, SO = ((NC - 2) & ~1) + 1;
                    float Ev = c[SE], Od = c[SO];
#pragma unroll
                    for (int i = SE - 2; i >= 0; i -= 2) Ev = fmaf(Ev, r2, c[i]);
#pragma unroll
                    for (int i = SO - 2; i >= 0; i -= 2) Od = fmaf(Od, r2, c[i]);
                    u = fmaf(Ev, rinv, Od);
                } else {
                    const float x = fmaf(r2, rinv, cen) * rsc;
                    float p = fmaf(c[NC - 1], x, c_next);
#pragma unroll
                    for (int i = NC - 3; i >= 0; --i) p = fmaf(p, x, c[i]);
                    u = p * rinv;
                }
            }
            auto add = [&](float &e, float q) {
                switch (s) {
                case 0: fmac_quad1<0>(e, q, u); break;
                case 1: fmac_quad1<1>(e, q, u); break;
                case 2: fmac_quad1<2>(e, q, u); break;
                default: fmac_quad1<3>(e, q, u); break;
                }
            };
            add(ea[0], pc.w);
            if (V > 1) add(ea[V - 1], q1);
        }
    };
    // two blocks per iteration, each block's point loaded one block ahead and its index two
    // blocks ahead (the padding keeps both in bounds); the two point registers alternate, so
    // no copies between blocks
    const int nb = K >> 2;
    int id = index(0);
    unsigned long long ma = __ballot(id < 0), mb;
    P4<float> pa = point(id), pb;
    float qa = charge1(id), qb = 0;
    id = index(1);
    int b = 0;
    for (; b + 2 <= nb; b += 2) {
        mb = __ballot(id < 0);
        pb = point(id);
        qb = charge1(id);
        id = index(b + 2);
        block(pa, qa, ma, 4 * b);
        ma = __ballot(id < 0);
        pa = point(id);
        qa = charge1(id);
        id = index(b + 3);
        block(pb, qb, mb, 4 * b + 4);
    }
    if (b < nb) block(pa, qa, ma, 4 * b);
    if (S > 1) {
#pragma unroll
        for (int v = 0; v < V; ++v) sum[v * (ne + 1) * 64] = ea[v];
        __syncthreads();
        if (w >= V) return;  // wave v adds component v
        double t = 0;
        for (int e = 0; e < ne; ++e) t += (double)sums[(w * (ne + 1) + e) * 64 + lane];
        if (active) pot_sorted[w * vs_pot + it.x + lane] += (float)t;
        return;
    }
#pragma unroll
    for (int v = 0; v < V; ++v)
        if (active) pot_sorted[v * vs_pot + it.x + lane] += (float)(acc[v] + (double)ea[v]);
}

// ------------------------------------------------ near field of many charge vectors (FP32)
// qv[i * VC + c] = charge c of sorted source i, for the VC vectors of a pass: vector v0 + c
// of Q (vector-major, N per vector; zero past the last vector).
template <int VC>
__global__ void k_gather_many(const double *__restrict__ Q, int n_vec, int v0, int n, const int *__restrict__ src_user,
                              int nsall, float *__restrict__ qv) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nsall) return;
    const int u = src_user[i];
#pragma unroll
    for (int c = 0; c < VC; ++c) qv[(size_t)i * VC + c] = v0 + c < n_vec ? (float)Q[(size_t)(v0 + c) * n + u] : 0.0f;
}

// ea[c] += q[c](lane 4 g + S) * u for 8 charges of a row's step: DPP-broadcast FMAs in one
// asm statement that starts with s_nop 1, the two wait states a DPP read needs after a VALU
// write of its source (the compiler does not check hazards inside inline asm).  ea and q point
// at 8 consecutive elements of register arrays (constant offsets once inlined).
#define PDMK_FMAC_QUAD(SEL)                                                                                    \
    asm("s_nop 1\n"                                                                                            \
        "v_fmac_f32_dpp %0, %8, %16 quad_perm:[" SEL "] row_mask:0xf bank_mask:0xf bound_ctrl:1\n"            \
        "v_fmac_f32_dpp %1, %9, %16 quad_perm:[" SEL "] row_mask:0xf bank_mask:0xf bound_ctrl:1\n"            \
        "v_fmac_f32_dpp %2, %10, %16 quad_perm:[" SEL "] row_mask:0xf bank_mask:0xf bound_ctrl:1\n"           \
        "v_fmac_f32_dpp %3, %11, %16 quad_perm:[" SEL "] row_mask:0xf bank_mask:0xf bound_ctrl:1\n"           \
        "v_fmac_f32_dpp %4, %12, %16 quad_perm:[" SEL "] row_mask:0xf bank_mask:0xf bound_ctrl:1\n"           \
        "v_fmac_f32_dpp %5, %13, %16 quad_perm:[" SEL "] row_mask:0xf bank_mask:0xf bound_ctrl:1\n"           \
        "v_fmac_f32_dpp %6, %14, %16 quad_perm:[" SEL "] row_mask:0xf bank_mask:0xf bound_ctrl:1\n"           \
        "v_fmac_f32_dpp %7, %15, %16 quad_perm:[" SEL "] row_mask:0xf bank_mask:0xf bound_ctrl:1\n"           \
        : "+v"(ea[0]), "+v"(ea[1]), "+v"(ea[2]), "+v"(ea[3]), "+v"(ea[4]), "+v"(ea[5]), "+v"(ea[6]), "+v"(ea[7]) \
        : "v"(q[0]), "v"(q[1]), "v"(q[2]), "v"(q[3]), "v"(q[4]), "v"(q[5]), "v"(q[6]), "v"(q[7]), "v"(u))

template <int S>
__device__ __forceinline__ void fmac_quad8(float *ea, const float *q, float u) {
    if constexpr (S == 0) PDMK_FMAC_QUAD("0,0,0,0");
    if constexpr (S == 1) PDMK_FMAC_QUAD("1,1,1,1");
    if constexpr (S == 2) PDMK_FMAC_QUAD("2,2,2,2");
    if constexpr (S == 3) PDMK_FMAC_QUAD("3,3,3,3");
}
#undef PDMK_FMAC_QUAD

// all VC charges of a step, 8 per asm block
template <int S, int VC>
__device__ __forceinline__ void fmac_quads(float (&ea)[VC], const float (&q)[VC], float u) {
#pragma unroll
    for (int v = 0; v < VC; v += 8) fmac_quad8<S>(ea + v, q + v, u);
}

// k_near_rows for VC charge vectors at once (a multiple of 8): the residual of each (target, source) pair is
// formed once and multiplied into VC sums.  pot_near[c * n + t] (c < vc) receives vector c's
// near field of sorted target t; each vector's sums are those of k_near_rows on that vector,
// bit for bit.
template <int NC, int VC>
__global__ __launch_bounds__(256) void k_near_rows_many(
    const P4<float> *__restrict__ src, const float *__restrict__ qv, const P4<float> *__restrict__ trg,
    const int4 *__restrict__ items, const int *__restrict__ l1_ptr, const P4<float> *__restrict__ geom,
    const int *__restrict__ rs_base, const int *__restrict__ rslot, const long long *__restrict__ wave_base,
    const int *__restrict__ steps, const float *__restrict__ coeffs, float *__restrict__ pot_near, int n, int vc,
    int item0, int item1, int ne_max) {
    static_assert(VC % 8 == 0, "the DPP FMA blocks take 8 vectors each");
    extern __shared__ float4 nf_lds[];
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int item = item0 + xcd_block(blockIdx.x, gridDim.x) * (blockDim.x >> 6) + w;
    if (item >= item1) return;  // whole wavefront (no workgroup barrier below)
    const int lane = threadIdx.x & 63, g = lane >> 2;
    const int4 it = items[item];
    float4 *geo = nf_lds + (size_t)w * (ne_max + 1) * 6;
    int *slots = reinterpret_cast<int *>(geo + 2 * (ne_max + 1));
    const int eb = l1_ptr[it.z], ne = l1_ptr[it.z + 1] - eb;
    for (int e = lane; e <= ne; e += 64) {
        const P4<float> gm = e < ne ? geom[eb + e] : P4<float>{0.0f, 0.0f, 0.0f, 0.0f};
        const float bs = gm.w;
        geo[2 * e] = make_float4(gm.x, gm.y, gm.z, bs * bs);
        geo[2 * e + 1] = make_float4(e < ne ? 2.0f / bs : 0.0f, -bs / 2.0f, 0.0f, 0.0f);
    }
    const int *rs = rslot + (size_t)rs_base[item] * NF_ROWS;
    for (int k = lane; k < (ne + 1) * NF_ROWS; k += 64) slots[k] = rs[k];
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const bool active = lane < it.y;
    const P4<float> me = active ? trg[it.x + lane] : P4<float>{1e18f, 1e18f, 1e18f, 0.0f};
    float c[NC];
#pragma unroll
    for (int i = 0; i < NC; ++i) c[i] = coeffs[i];
    float c_next;  // as in k_near_rows
    asm("v_mov_b32 %0, %1" : "=v"(c_next) : "s"(c[NC - 2]));
    float tx = 0, ty = 0, tz = 0, d2max = 0, rsc = 0, cen = 0;
    int end = 0, ns = 0;
    double acc[VC];
    float ea[VC];
#pragma unroll
    for (int v = 0; v < VC; ++v) {
        acc[v] = 0;
        ea[v] = 0;
    }
    auto enter = [&]() {
#pragma unroll
        for (int v = 0; v < VC; ++v) {
            acc[v] += (double)ea[v];
            ea[v] = 0;
        }
        const int sv = slots[ns * NF_ROWS + g];
        ++ns;
        const int o = sv & 255;
        end = sv >> 8;
        const float4 a = geo[2 * o], b = geo[2 * o + 1];
        tx = me.x + a.x;
        ty = me.y + a.y;
        tz = me.z + a.z;
        d2max = a.w;
        rsc = b.x;
        cen = b.y;
    };
    enter();
    const int K = it.w;
    const int *sp = steps + wave_base[item] + lane;
    int id = sp[0];
    P4<float> pc = nf_load_u32<P4<float>>(src, (unsigned)id * 16u);
    float qc[VC];
#pragma unroll
    for (int v = 0; v < VC; v += 4)
        *reinterpret_cast<float4 *>(&qc[v]) = nf_load_u32<float4>(qv + v, (unsigned)id * (unsigned)(VC * sizeof(float)));
    id = sp[64];
    for (int k = 0; k < K; k += 4) {
        const P4<float> pn = nf_load_u32<P4<float>>(src, (unsigned)id * 16u);
        float qn[VC];
#pragma unroll
        for (int v = 0; v < VC; v += 4)
            *reinterpret_cast<float4 *>(&qn[v]) = nf_load_u32<float4>(qv + v, (unsigned)id * (unsigned)(VC * sizeof(float)));
        id = sp[(size_t)(k + 8) * NF_ROWS];
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            if (k + s >= end) enter();
            float px, py, pz;
            switch (s) {
            case 0: px = quad_bcast<0>(pc.x); py = quad_bcast<0>(pc.y); pz = quad_bcast<0>(pc.z); break;
            case 1: px = quad_bcast<1>(pc.x); py = quad_bcast<1>(pc.y); pz = quad_bcast<1>(pc.z); break;
            case 2: px = quad_bcast<2>(pc.x); py = quad_bcast<2>(pc.y); pz = quad_bcast<2>(pc.z); break;
            default: px = quad_bcast<3>(pc.x); py = quad_bcast<3>(pc.y); pz = quad_bcast<3>(pc.z); break;
            }
            const float dx = px - tx, dy = py - ty, dz = pz - tz;
            const float r2 = fmaf(dx, dx, fmaf(dy, dy, dz * dz));
            float u = 0;
            if (r2 < d2max && r2 > 1e-30f) {
                const float rinv = rsqrt_full<float>(r2);
                const float x = fmaf(r2, rinv, cen) * rsc;
                float p = fmaf(c[NC - 1], x, c_next);
#pragma unroll
                for (int i = NC - 3; i >= 0; --i) p = fmaf(p, x, c[i]);
                u = p * rinv;
            }
            switch (s) {
            case 0: fmac_quads<0>(ea, qc, u); break;
            case 1: fmac_quads<1>(ea, qc, u); break;
            case 2: fmac_quads<2>(ea, qc, u); break;
            default: fmac_quads<3>(ea, qc, u); break;
            }
        }
        pc = pn;
#pragma unroll
        for (int v = 0; v < VC; ++v) qc[v] = qn[v];
    }
    if (active) {
#pragma unroll
        for (int v = 0; v < VC; ++v)
            if (v < vc) pot_near[(size_t)v * n + it.x + lane] = (float)(acc[v] + (double)ea[v]);
    }
}

// The FP64 row kernel (NC coefficients, x form).  The same step lists and slots; a row's 4
// points of a block reach its lanes through LDS (64-bit DPP has no quad broadcast): each lane
// writes the point it loaded, then every lane reads its row's point of the step.  Per
// wavefront LDS: 64 points (2 KiB), then (ne_max + 1) entries x 48 bytes of geometry and
// (ne_max + 1) x 16 slots, decoded in LDS as in the FP32 kernel.  The same loop structure as
// the FP32 kernel (two blocks per iteration, scalar entry-switch tests).  Bit-identical to
// k_near_field<double, NC, false> for the same reason as the FP32 kernel.
__host__ __device__ inline size_t near_rows64_lds_per_wave(int ne_max) {
    return 64 * 2 * sizeof(double2) + (size_t)(ne_max + 1) * 3 * sizeof(double2) + (size_t)(ne_max + 1) * NF_ROWS * 4;
}

template <int NC, int S>
__global__ __launch_bounds__(1024) void k_near_rows64(const P4<double> *__restrict__ src,
                                                      const P4<double> *__restrict__ trg,
                                                      const int4 *__restrict__ items, const int *__restrict__ l1_ptr,
                                                      const P4<double> *__restrict__ geom,
                                                      const int *__restrict__ rs_base, const int *__restrict__ rslot,
                                                      const long long *__restrict__ wave_base,
                                                      const int *__restrict__ steps, const double *__restrict__ coeffs,
                                                      double *__restrict__ pot_sorted, int item0, int item1, int ne_max,
                                                   long long vs_src = 0, long long vs_pot = 0) {
    src += (long long)blockIdx.z * vs_src;  // component blockIdx.z of a quasi-periodic pass
    pot_sorted += (long long)blockIdx.z * vs_pot;
    extern __shared__ double2 nf_lds64[];
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int item = S > 1 ? (item0 + (int)blockIdx.x) * S + w
                           : item0 + xcd_block(blockIdx.x, gridDim.x) * (blockDim.x >> 6) + w;
    if (S == 1 && item >= item1) return;  // whole wavefront (no workgroup barrier below)
    const int lane = threadIdx.x & 63, g = lane >> 2;
    const int4 it = items[item];  // (first target, count, target-leaf list index, K)
    double2 *pts = reinterpret_cast<double2 *>(reinterpret_cast<char *>(nf_lds64) + (size_t)w * near_rows64_lds_per_wave(ne_max));
    double2 *geo = pts + 128;
    int *slots = reinterpret_cast<int *>(geo + 3 * (ne_max + 1));
    const int eb = l1_ptr[it.z], ne = l1_ptr[it.z + 1] - eb;
    // S > 1: the entries' sums [ne + 1][64]
    double *sums = reinterpret_cast<double *>(reinterpret_cast<char *>(nf_lds64) + (size_t)S * near_rows64_lds_per_wave(ne_max));
    if (S > 1) {
        for (int k = threadIdx.x; k < ne * 64; k += 64 * S) sums[k] = 0;
        __syncthreads();
    }
    for (int e = lane; e <= ne; e += 64) {
        const P4<double> gm = e < ne ? geom[eb + e] : P4<double>{0.0, 0.0, 0.0, 0.0};
        const double bs = gm.w;
        geo[3 * e] = make_double2(gm.x, gm.y);
        geo[3 * e + 1] = make_double2(gm.z, bs * bs);
        geo[3 * e + 2] = make_double2(e < ne ? 2.0 / bs : 0.0, -bs / 2.0);
    }
    const int *rs = rslot + (size_t)rs_base[item] * NF_ROWS;
    const unsigned geo_off = (unsigned)((const char *)geo - (const char *)nf_lds64);
    const int n_slots = S > 1 ? rs_base[item + 1] - rs_base[item] : ne + 1;
    for (int k = lane; k < n_slots * NF_ROWS; k += 64) {
        const int v = rs[k];
        slots[k] = (int)(((unsigned)min(v >> 8, 0xffff) << 16) | (geo_off + 48u * (unsigned)(v & 255)));
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const bool active = lane < it.y;
    const P4<double> me = active ? trg[it.x + lane] : P4<double>{1e18, 1e18, 1e18, 0.0};
    double c[NC];
#pragma unroll
    for (int i = 0; i < NC; ++i) c[i] = coeffs[i];
    const double ctop = c[NC - 1] + (double)vgpr_zero();  // leading coefficient in a VGPR (see k_near_field)
    double tx = 0, ty = 0, tz = 0, d2max = 0, rsc = 0, cen = 0;
    int end = 0;
    const int *slot = slots + g;  // the row's next slot
    double acc = 0, ea = 0;
    double *sum = sums + (size_t)ne * 64 + lane;  // the current entry's (row ne: none)
    auto enter = [&]() {  // the row's next non-empty entry (or the terminator)
        if (S > 1) *sum = ea;
        else acc += ea;
        ea = 0;
        const unsigned v = (unsigned)*slot;
        slot += NF_ROWS;
        end = (int)(v >> 16);
        if (S > 1) sum = sums + ((v & 0xffffu) - geo_off) / 48u * 64u + lane;
        const double2 *ge = reinterpret_cast<const double2 *>(reinterpret_cast<const char *>(nf_lds64) + (v & 0xffffu));
        const double2 a = ge[0], b = ge[1], cc = ge[2];
        tx = me.x + a.x;
        ty = me.y + a.y;
        tz = me.z + b.x;
        d2max = b.y;
        rsc = cc.x;
        cen = cc.y;
    };
    enter();
    const int K = it.w;
    const int *sb = steps + wave_base[item];
    auto index = [&](int b) { return nf_load_u32<int>(sb + (size_t)b * 64, (unsigned)lane * 4u); };
    auto point = [&](int id) { return nf_load_u32<P4<double>>(src, (unsigned)id * 32u); };
    // m: ballot of the block's entry flags, bit 4 g + s = row g switches entries at step s
    auto block = [&](const P4<double> &pc, unsigned long long m, int k) {
        pts[2 * lane] = make_double2(pc.x, pc.y);
        pts[2 * lane + 1] = make_double2(pc.z, pc.w);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            // the wave-wide switch test is scalar; the empty asm keeps the per-lane test inside
            if ((m >> s) & 0x1111111111111111ull) {
                asm volatile("");
                if (k + s >= end) enter();
            }
            const double2 a = pts[2 * (4 * g + s)], b = pts[2 * (4 * g + s) + 1];
            // (source - target: the negated difference, exactly, so r^2 is the same)
            const double dx = a.x - tx, dy = a.y - ty, dz = b.x - tz;
            const double r2 = fma(dx, dx, fma(dy, dy, dz * dz));
            if (r2 < d2max && r2 > 1e-30) {
                const double rinv = rsqrt_full<double>(r2);
                const double x = fma(r2, rinv, cen) * rsc;
                double p = ctop;
#pragma unroll
                for (int i = NC - 2; i >= 0; --i) p = fma(p, x, c[i]);
                ea = fma(p * rinv, b.y, ea);
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();  // every lane has read the block before it is overwritten
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    // two blocks per iteration, points one block ahead, indices two (see k_near_rows)
    const int nb = K >> 2;
    int id = index(0);
    unsigned long long ma = __ballot(id < 0), mb;
    P4<double> pa = point(id), pb;
    id = index(1);
    int b = 0;
    for (; b + 2 <= nb; b += 2) {
        mb = __ballot(id < 0);
        pb = point(id);
        id = index(b + 2);
        block(pa, ma, 4 * b);
        ma = __ballot(id < 0);
        pa = point(id);
        id = index(b + 3);
        block(pb, mb, 4 * b + 4);
    }
    if (b < nb) block(pa, ma, 4 * b);
    if (S > 1) {
        *sum = ea;
        __syncthreads();
        if (w > 0) return;
        for (int e = 0; e < ne; ++e) acc += sums[e * 64 + lane];
    } else {
        acc += ea;
    }
    if (active) pot_sorted[it.x + lane] += acc;
}

template <class R>
__global__ void k_fill(R *__restrict__ p, R v, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

// ------------------------------------------------------------------ far field
// Half-space modes with nonzero weight come in lines of constant (j, k) with i contiguous.
// All far-field arithmetic is FP64, on the matrix cores: along i the phases are real,
//   sum_i f_i e^{-+ i i th1} = sum_{i >= 0} (combinations of f_i, f_-i) x (cos i th1, sin i th1),
// so both directions are products of a real table trig[point][2 i + (0 cos, 1 sin)] with the
// lines' complex parts, 2 multiply-adds per mode and point where a recurrence per mode takes
// 6 (structure factors) and a Horner step 4 (evaluation).  Lines are sorted by their largest
// |i| and taken 16 at a time (line tiles), so that a tile only spends the columns it needs.
// The rows of a tile of points (trig along axis 0, e^{i m th} for m >= 0 along axes 1 and 2:
// negative m by conjugation) are tabulated in LDS by recurrence from one sincos per axis.
// The vector kernels these replace ran a lane per mode chunk or per point and were bound by
// latency (one point per lane of a 4-workgroup launch at N = 1e3) and FP64 issue.
constexpr int FF_UNITS = 16;  // most (line tile, 16 trig columns) units of a structure-factor workgroup
constexpr int FF_MANY = 2;    // vectors per workgroup of a many-vector launch

__device__ __forceinline__ double2 cmul(double2 a, double2 b) {
    return make_double2(fma(a.x, b.x, -a.y * b.y), fma(a.x, b.y, a.y * b.x));
}

// Index bounds of the listed modes: |i| <= I, |j| <= J, |k| <= K.  LDS row of a point:
// ts() doubles of trig (an odd count: the evaluation reads 16 points' rows at once), then
// J + 1 and K + 1 complex phases.
struct FfDims {
    int I, J, K;
    __host__ __device__ int ts() const { return 2 * I + 3; }
    __host__ __device__ size_t lds_bytes(int tp) const {
        return (size_t)tp * (sizeof(double) * ts() + sizeof(double2) * (J + 1 + K + 1));
    }
};

// LDS tables of points p0 .. p0 + tp - 1 (phases e^{sgn i m th}; points past n: theta 0).  The
// pad column of trig is 0.
__device__ __forceinline__ void ff_tables(double *trig, double2 *E2, double2 *E3, const double *__restrict__ theta, int n,
                                          int p0, int tp, FfDims d, double sgn) {
    for (int t = threadIdx.x; t < tp * 3; t += blockDim.x) {
        const int pp = t % tp, ax = t / tp, gp = p0 + pp;
        double s1, c1;
        sincos(gp < n ? theta[3 * (size_t)gp + ax] : 0.0, &s1, &c1);
        if (ax == 0) {
            double *row = trig + (size_t)pp * d.ts();
            double2 cur = make_double2(1, 0);
            for (int m = 0; m <= d.I; ++m) {
                row[2 * m] = cur.x;
                row[2 * m + 1] = cur.y;
                cur = cmul(cur, make_double2(c1, s1));
            }
            row[2 * d.I + 2] = 0;
        } else {
            const int cnt = ax == 1 ? d.J : d.K;
            double2 *row = (ax == 1 ? E2 : E3) + (size_t)pp * (cnt + 1);
            const double2 step = make_double2(c1, sgn * s1);
            double2 cur = make_double2(1, 0);
            for (int m = 0; m <= cnt; ++m) {
                row[m] = cur;
                cur = cmul(cur, step);
            }
        }
    }
}

// Partial structure factors per workgroup column of points:
//   Sp[blk][m] = sum_{points of blk} q e^{-i(i th1 + j th2 + k th3)}.
// Unit (line tile, ct): the 16 x 16 products of 16 lines' a = e^{-i(j th2 + k th3)} (real and
// imaginary part, one accumulator each) with 16 trig columns times q, summed over points 4 at a time
// by v_mfma_f64_16x16x4f64 (lane l supplies A[l % 16][l / 16] = its line's a at point l / 16 and
// B[l / 16][l % 16] = q trig, and holds D[l / 16 + 4 e][l % 16]).  A wave owns U units (those
// past the last are formed and not stored: with a test per unit the compiler cannot have the
// LDS reads of all U in flight), a workgroup 4 U (grid y).  At the end the cos and sin columns
// of a line (neighbouring lanes) combine into modes +i and -i.  Workgroup z of a many-vector
// launch takes vectors V z .. V z + V - 1 (< nv; vector v's charges at q + v vs_q, its sums at
// Sp + v vs_sp) on one set of tables and phases; each vector's sums are those of a one-vector
// launch, bit for bit.
//
// CPLX (quasi-periodic, V = 1): charges q e^{-i bx} and lines over the whole mode box.
template <int U, int V, bool CPLX>
__global__ __launch_bounds__(256, 2) void k_ff_structure(const double *__restrict__ theta, const double *__restrict__ q,
                                                       const double *__restrict__ bx, int n,
                                                       int tp, FfDims d, const int4 *__restrict__ lines,
                                                       const int *__restrict__ line_m0, const int2 *__restrict__ units,
                                                       int n_units, int n_modes, double2 *__restrict__ Sp,
                                                       long long vs_q = 0, long long vs_sp = 0, int nv = 1) {
    extern __shared__ double2 ff_lds[];
    static_assert(!CPLX || V == 1, "complex charges: one vector");
    __shared__ double Qs[CPLX ? 2 : V][32];
    const int v0 = blockIdx.z * V;
    double *trig = reinterpret_cast<double *>(ff_lds);
    const int ts = d.ts();
    double2 *E2 = reinterpret_cast<double2 *>(trig + (size_t)tp * ts), *E3 = E2 + (size_t)tp * (d.J + 1);
    const int lane = threadIdx.x & 63, kk = lane >> 4, jj = lane & 15;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int u0 = (blockIdx.y * 4 + w) * U;
    int o2[U], o3[U], oc[U];  // LDS offsets of the lane's j and k phases, and of its trig column
    double s2[U], s3[U];      // signs of j and k
    c2p_d4 are[V][U], aim[V][U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int2 un = units[min(u0 + u, n_units - 1)];
        const int4 ln = lines[un.x * 16 + jj];
        o2[u] = abs(ln.x);
        o3[u] = abs(ln.y);
        s2[u] = ln.x < 0 ? -1.0 : 1.0;
        s3[u] = ln.y < 0 ? -1.0 : 1.0;
        oc[u] = 16 * un.y + jj;
#pragma unroll
        for (int v = 0; v < V; ++v) are[v][u] = aim[v][u] = c2p_d4{0, 0, 0, 0};
    }
    for (int p0 = blockIdx.x * tp; p0 < n; p0 += gridDim.x * tp) {
        __syncthreads();
        ff_tables(trig, E2, E3, theta, n, p0, tp, d, -1.0);
        // (from the last threads down: the first ones are busy with the tables)
        for (int t = 255 - (int)threadIdx.x; t < tp * V; t += 256) {
            const int pp = t % tp, v = t / tp;
            if constexpr (CPLX) {
                double sn = 0, cs = 0;
                if (p0 + pp < n) sincos(bx[p0 + pp], &sn, &cs);
                const double qp = p0 + pp < n ? q[p0 + pp] : 0.0;
                Qs[0][pp] = qp * cs;
                Qs[CPLX][pp] = -qp * sn;
                continue;
            }
            Qs[v][pp] = p0 + pp < n && v0 + v < nv ? q[(long long)(v0 + v) * vs_q + p0 + pp] : 0.0;
        }
        __syncthreads();
        for (int k0 = 0; k0 < tp; k0 += 4) {  // (a wave-uniform count: the accumulators stay in place)
            const int p = k0 + kk;
            const double *tr = trig + (size_t)p * ts;
            const double2 *r2 = E2 + (size_t)p * (d.J + 1), *r3 = E3 + (size_t)p * (d.K + 1);
            double b[U];
            double2 x[U], y[U];
            double qq[V];
#pragma unroll
            for (int v = 0; v < V; ++v) qq[v] = Qs[v][p];
            const double qi = CPLX ? Qs[CPLX][p] : 0.0;
#pragma unroll
            for (int u = 0; u < U; ++u) {
                b[u] = tr[oc[u]];
                x[u] = r2[o2[u]];
                y[u] = r3[o3[u]];
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const double xi = s2[u] * x[u].y, yi = s3[u] * y[u].y;
                const double ar = fma(x[u].x, y[u].x, -xi * yi), ai = fma(x[u].x, yi, xi * y[u].x);
                if constexpr (CPLX) {
                    are[0][u] = __builtin_amdgcn_mfma_f64_16x16x4f64(fma(qq[0], ar, -qi * ai), b[u], are[0][u], 0, 0, 0);
                    aim[0][u] = __builtin_amdgcn_mfma_f64_16x16x4f64(fma(qq[0], ai, qi * ar), b[u], aim[0][u], 0, 0, 0);
                    continue;
                }
#pragma unroll
                for (int v = 0; v < V; ++v) {
                    const double qb = qq[v] * b[u];
                    are[v][u] = __builtin_amdgcn_mfma_f64_16x16x4f64(ar, qb, are[v][u], 0, 0, 0);
                    aim[v][u] = __builtin_amdgcn_mfma_f64_16x16x4f64(ai, qb, aim[v][u], 0, 0, 0);
                }
            }
        }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
        if (u0 + u >= n_units) break;
        const int2 un = units[u0 + u];
        const int c = 16 * un.y + jj, i = (c & 1) ? -(c >> 1) : (c >> 1);  // even: cos, mode +i; odd: sin, mode -i
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int line = un.x * 16 + kk + 4 * e;
            const int4 ln = lines[line];
            const bool mode = i >= ln.z && i <= ln.w && !((c & 1) && i == 0);
            double2 *out = Sp + (size_t)blockIdx.x * n_modes + line_m0[line] + i - ln.z;
#pragma unroll
            for (int v = 0; v < V; ++v) {
                const double mr = are[v][u][e], mi = aim[v][u][e], pr = __shfl_xor(mr, 1), pi = __shfl_xor(mi, 1);
                // S(+i) = C - i D, S(-i) = C + i D (C the cos, D the sin column)
                if (mode && v0 + v < nv)
                    out[(long long)(v0 + v) * vs_sp] = (c & 1) ? make_double2(pr - mi, pi + mr) : make_double2(mr + pi, mi - pr);
            }
        }
    }
}

// Column sums of the partial structure factors, weighted, as the evaluation's operands:
// with T(+-i) = w S(+-i), line (j, k) contributes Re(e^{i(j th2 + k th3)} sum_i (Gc cos i th1 +
// Gs sin i th1)), Gc = T(i) + T(-i), Gs = i (T(i) - T(-i)).  Tile t's G starts at info[t].y:
// [ks][re, im][64], column 4 ks + l / 16 of line l % 16 at lane l.  One workgroup per line, its
// modes contiguous: 32 modes x 16 groups of columns at a time, the groups added in order, the
// weighted sums of the line kept in LDS for the (+i, -i) pairs.  (32 modes x 8 groups per
// workgroup, one thread per 64 columns, left 44 workgroups to read all partial sums: 21 us at
// N = 1e4, 110 us at 2.5e5 beside the near field.)
__global__ __launch_bounds__(512) void k_ff_reduce(const double2 *__restrict__ Sp, int nblk, const double *__restrict__ w,
                                                   const int4 *__restrict__ lines, const int *__restrict__ line_m0,
                                                   const int2 *__restrict__ info, int n_modes, double *__restrict__ G,
                                                   long long vs_sp = 0, long long vs_g = 0) {
    extern __shared__ double2 ff_lds[];
    double2 *part = ff_lds, *T = ff_lds + 512;  // T[mode of the line]
    const int4 ln = lines[blockIdx.x];
    const int len = ln.w - ln.z + 1, m0 = line_m0[blockIdx.x];
    if (len <= 0) return;  // padding line: its G stays zero
    Sp += (long long)blockIdx.z * vs_sp + m0;
    const int l = threadIdx.x & 31, g = threadIdx.x >> 5;
    for (int c = 0; c < len; c += 32) {
        double2 a = make_double2(0, 0);
        if (c + l < len) {
#pragma unroll 4
            for (int k = g; k < nblk; k += 16) {
                const double2 x = Sp[(size_t)k * n_modes + c + l];
                a.x += x.x;
                a.y += x.y;
            }
        }
        part[threadIdx.x] = a;
        __syncthreads();
        if (g == 0 && c + l < len) {
            double2 t = make_double2(0, 0);
#pragma unroll
            for (int k = 0; k < 16; ++k) {
                t.x += part[32 * k + l].x;
                t.y += part[32 * k + l].y;
            }
            const double wm = w[m0 + c + l];
            T[c + l] = make_double2(t.x * wm, t.y * wm);
        }
        __syncthreads();
    }
    const int2 inf = info[blockIdx.x >> 4];
    G += (long long)blockIdx.z * vs_g + inf.y;
    for (int i = threadIdx.x; i <= inf.x; i += 512) {
        double2 u = make_double2(0, 0), v = make_double2(0, 0);
        if (i >= ln.z && i <= ln.w) u = T[i - ln.z];
        if (i > 0 && -i >= ln.z && -i <= ln.w) v = T[-i - ln.z];
        double *o = G + (size_t)(i >> 1) * 128 + (i & 1) * 32 + (blockIdx.x & 15);  // columns 2 i, 2 i + 1
        o[0] = u.x + v.x;
        o[64] = u.y + v.y;
        o[16] = v.y - u.y;
        o[64 + 16] = u.x - v.x;
    }
}

// far[u] = sum_m Re( S[m] e^{+i(i th1 + j th2 + k th3)} ).  Per line tile the products
// D = trig x G (points by lines, real and imaginary part) on the matrix cores, then
// Re(e^{i(j th2 + k th3)} D) added up per point.  A workgroup takes 16 RT points; its 4 waves
// share the line tiles, so that also a few hundred points fill several CUs, and their sums
// are added in wave order.  Workgroup z of a many-vector launch evaluates vectors V z .. (< nv;
// G + v vs_g, output at far + v vs_far) on one set of tables and phases, each as a one-vector
// launch does, bit for bit.
// CPLX: far holds complex values, e^{i bx} sum_m S[m] e^{i m.th}.
template <int RT, int V, bool CPLX>
__global__ __launch_bounds__(256, 2) void k_ff_eval(const double *__restrict__ theta, const double *__restrict__ bx, int n,
                                                 FfDims d,
                                                 const int4 *__restrict__ lines, const int2 *__restrict__ info, int n_lt,
                                                 const double *__restrict__ G, double *__restrict__ far,
                                                 long long vs_g = 0, long long vs_far = 0, int nv = 1) {
    extern __shared__ double2 ff_lds[];
    constexpr int TP = 16 * RT;
    static_assert(!CPLX || V == 1, "complex charges: one vector");
    constexpr int VO = CPLX ? 2 : V;  // sums per point
    __shared__ double red[VO][4][TP];
    const int v0 = blockIdx.z * V;
    double *trig = reinterpret_cast<double *>(ff_lds);
    const int ts = d.ts();
    double2 *E2 = reinterpret_cast<double2 *>(trig + (size_t)TP * ts), *E3 = E2 + (size_t)TP * (d.J + 1);
    const int p0 = blockIdx.x * TP;
    ff_tables(trig, E2, E3, theta, n, p0, TP, d, 1.0);
    __syncthreads();
    const int lane = threadIdx.x & 63, kk = lane >> 4, jj = lane & 15;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    double acc[VO][RT][4];
#pragma unroll
    for (int v = 0; v < VO; ++v)
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[v][rt][e] = 0;
    for (int lt = w; lt < n_lt; lt += 4) {
        const int2 inf = info[lt];
        const int nks = (inf.x + 2) >> 1;  // 4 columns each: 2 (imax + 1), rounded up
        const int4 ln = lines[lt * 16 + jj];
        c2p_d4 dr[V][RT], di[V][RT];
        const double *tr = trig + (size_t)jj * ts + kk;
#pragma unroll
        for (int v = 0; v < V; ++v) {
            // (a vector past nv repeats vector v0 and stores nothing)
            const double *g = G + (long long)(v0 + (v0 + v < nv ? v : 0)) * vs_g + inf.y + lane;
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) dr[v][rt] = di[v][rt] = c2p_d4{0, 0, 0, 0};
            double br = g[0], bi = g[64];
            for (int ks = 0; ks < nks; ++ks) {
                // the next step's operands (the last step reads the table's padding)
                const double nr = g[(size_t)(ks + 1) * 128], ni = g[(size_t)(ks + 1) * 128 + 64];
#pragma unroll
                for (int rt = 0; rt < RT; ++rt) {
                    const double a = tr[(size_t)rt * 16 * ts + 4 * ks];
                    dr[v][rt] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, br, dr[v][rt], 0, 0, 0);
                    di[v][rt] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, bi, di[v][rt], 0, 0, 0);
                }
                br = nr;
                bi = ni;
            }
        }
        const int o2 = abs(ln.x), o3 = abs(ln.y);
        const double s2 = ln.x < 0 ? -1.0 : 1.0, s3 = ln.y < 0 ? -1.0 : 1.0;
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int p = 16 * rt + kk + 4 * e;
                const double2 x = E2[(size_t)p * (d.J + 1) + o2], y = E3[(size_t)p * (d.K + 1) + o3];
                const double xi = s2 * x.y, yi = s3 * y.y;
                const double ar = fma(x.x, y.x, -xi * yi), ai = fma(x.x, yi, xi * y.x);
#pragma unroll
                for (int v = 0; v < V; ++v)
                    acc[v][rt][e] = fma(ar, dr[v][rt][e], fma(-ai, di[v][rt][e], acc[v][rt][e]));
                if constexpr (CPLX) acc[1][rt][e] = fma(ar, di[0][rt][e], fma(ai, dr[0][rt][e], acc[1][rt][e]));
            }
    }
#pragma unroll
    for (int v = 0; v < VO; ++v)
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                double t = acc[v][rt][e];
#pragma unroll
                for (int m = 8; m >= 1; m >>= 1) t += __shfl_xor(t, m, 16);
                if (jj == 0) red[v][w][16 * rt + kk + 4 * e] = t;
            }
    __syncthreads();
    for (int t = threadIdx.x; t < TP * V; t += blockDim.x) {
        const int v = t / TP, p = t % TP;
        if constexpr (CPLX) {
            if (p0 + p >= n) continue;
            double sn, cs;
            sincos(bx[p0 + p], &sn, &cs);
            reinterpret_cast<double2 *>(far)[p0 + p] =
                cmul(make_double2(red[0][0][p] + red[0][1][p] + red[0][2][p] + red[0][3][p],
                                  red[1][0][p] + red[1][1][p] + red[1][2][p] + red[1][3][p]),
                     make_double2(cs, sn));
            continue;
        }
        if (p0 + p < n && v0 + v < nv)
            far[(long long)(v0 + v) * vs_far + p0 + p] = red[v][0][p] + red[v][1][p] + red[v][2][p] + red[v][3][p];
    }
}

// ------------------------------------------------------------------ far field by NUFFT
// Spreading, grid DFTs, deconvolution and interpolation of the non-uniform FFT evaluation of
// the same truncated Fourier sum (kernel values and point order prepared on the host).
// Grid layout [g2][g1][g0] (axis 0 fastest); mode box [k2][k1][k0], k = m + M/2.

// Lane l of a wavefront owns the kernel offsets (dy, dz) = (j % W, j / W), j = l + 64 ps
// (NP passes when W^2 > 64), and keeps its subgrid row (y, z) = (by + dy, bz + dz), the E
// cells along x, in registers.  A point's kernel along x is stored already placed in the row
// (phi_x at bx .. bx + W - 1, zeros elsewhere), held by lanes 0..E-1 of every 16-lane row and
// broadcast with DPP, so every point costs E FMAs per pass whatever its base bx; ky[dy],
// kz[dz], the charge and the row id are per-lane loads, issued D points ahead.
template <int W, int E> struct NufftCfg {
    static constexpr int NP = (W * W + 63) / 64;
    static constexpr int KS = E + 2 * W;  // kernel values per point
    static constexpr int D = NP == 1 ? 8 : 4;
};

template <int NP> struct NuPoint {
    double ka, kb, q, y[NP], z[NP];
    int pb;
};

// A zero the compiler cannot see through: indexing a uniform load with it keeps the load on
// the vector path, whose in-order completion lets the loads of later points stay in flight
// (a scalar load would need a full wait on every use).
__device__ __forceinline__ int nu_vzero() {
    int z;
    asm volatile("v_mov_b32 %0, 0" : "=v"(z));
    return z;
}

// Loads point p (kernel row, ky[dy], kz[dz], charge if Q, packed base); vz = nu_vzero().
template <int W, int E, bool Q, int NP>
__device__ __forceinline__ void nu_load(NuPoint<NP> &s, const double *__restrict__ kval, const double *__restrict__ qs,
                                        const int *__restrict__ pbase, int p, int rl, int vz, const int (&oy)[NP],
                                        const int (&oz)[NP]) {
    constexpr int KS = NufftCfg<W, E>::KS;
    const double *kv = kval + (size_t)p * KS;
    s.ka = kv[min(rl, KS - 1)];
    s.kb = E > 16 ? kv[min(16 + rl, KS - 1)] : 0.0;
#pragma unroll
    for (int ps = 0; ps < NP; ++ps) {
        s.y[ps] = kv[E + oy[ps]];
        s.z[ps] = kv[E + W + oz[ps]];
    }
    s.q = Q ? qs[p + vz] : 0.0;
    s.pb = pbase[p + vz];
}

// ---- per-point plan data of the NUFFT (built once per tree)
struct NufftGridArgs {
    int n[3], ntile[3], T, lo, B, W, E, KS;
    double h[3], beta;
};

__device__ __forceinline__ double nu_es_kernel(double z, double beta) {
    return fabs(z) < 1.0 ? exp(beta * (sqrt(1.0 - z * z) - 1.0)) : 0.0;
}

// Grid coordinate x in [0, n), tile coordinate and first grid point of the support along
// axis d of the point with angle theta.
__device__ __forceinline__ void nu_axis(double theta, const NufftGridArgs &a, int d, double &x, int &tc, int &g0) {
    const int n = a.n[d];
    x = theta / a.h[d];
    if (x < 0) x = 0;
    if (x >= n) x = nextafter((double)n, 0.0);
    tc = min(n - 1, (int)floor(x)) / a.T;
    g0 = (int)floor(x - 0.5 * a.W) + 1;
}

// key[u] = tile B^3 + (bz B + by) B + bx; bad[0] = 1 if a base leaves [0, B).
__global__ __launch_bounds__(256) void k_nufft_keys(const double *__restrict__ theta, int n, NufftGridArgs a,
                                                    int *__restrict__ key, int *__restrict__ bad) {
    const int u = blockIdx.x * blockDim.x + threadIdx.x;
    if (u >= n) return;
    int tc[3], b[3];
    for (int d = 0; d < 3; ++d) {
        double x;
        int g0;
        nu_axis(theta[3 * (size_t)u + d], a, d, x, tc[d], g0);
        b[d] = g0 - a.T * tc[d] - a.lo;
        if (b[d] < 0 || b[d] >= a.B) {
            bad[0] = 1;
            b[d] = 0;
        }
    }
    const int tile = (tc[2] * a.ntile[1] + tc[1]) * a.ntile[0] + tc[0];
    key[u] = tile * a.B * a.B * a.B + (b[2] * a.B + b[1]) * a.B + b[0];
}

// Plan-order rows: kval[i] = (phi_x placed at bx .. bx+W-1 of the E-cell row, phi_y, phi_z)
// and pbase[i] for the point u = order[i].
__global__ __launch_bounds__(256) void k_nufft_rows(const double *__restrict__ theta, const int *__restrict__ order, int n,
                                                    NufftGridArgs a, double *__restrict__ kval, int *__restrict__ pbase) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int u = order[i];
    double *row = kval + (size_t)i * a.KS;
    int b[3];
    for (int d = 0; d < 3; ++d) {
        double x;
        int tc, g0;
        nu_axis(theta[3 * (size_t)u + d], a, d, x, tc, g0);
        b[d] = min(max(g0 - a.T * tc - a.lo, 0), a.B - 1);
        double *dst = d == 0 ? row + b[0] : row + a.E + (d - 1) * a.W;
        if (d == 0)
            for (int k = 0; k < a.E; ++k) row[k] = 0.0;
        for (int k = 0; k < a.W; ++k) dst[k] = nu_es_kernel((x - (g0 + k)) / (0.5 * a.W), a.beta);
    }
    pbase[i] = b[0] | (b[1] << 8) | (b[2] << 16);
}

// cnt[tile]++ for every point (keys of k_nufft_keys).
__global__ __launch_bounds__(256) void k_nufft_tile_hist(const int *__restrict__ key, int n, int B3, int *__restrict__ cnt) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) atomicAdd(&cnt[key[i] / B3], 1);
}

// qs[i] = q[order[i]]: the charges in plan order.
__global__ __launch_bounds__(256) void k_nufft_permute(const double *__restrict__ q, const int *__restrict__ order, int n,
                                                       double *__restrict__ qs) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) qs[i] = q[order[i]];
}

// One wavefront per work unit (the points of one tile, or a part of them).  The lanes sum
// q phi_x phi_y phi_z over the points of a subgrid row (consecutive points with one (by, bz))
// in registers and add the row into the tile subgrid in LDS when the row changes; the
// subgrid (E^3, compact) goes to scratch[slot].  The sum order is fixed by the plan, so the
// result is deterministic.
template <int W, int E>
__global__ __launch_bounds__(64) void k_nufft_spread(const int *__restrict__ unit_ptr, const int *__restrict__ unit_slot,
                                                     const double *__restrict__ kval, const double *__restrict__ qs,
                                                     const int *__restrict__ pbase, int SY, int SZ,
                                                     double *__restrict__ scratch) {
    using C = NufftCfg<W, E>;
    constexpr int NP = C::NP, D = C::D;
    extern __shared__ double nu_lds[];
    double *sub = nu_lds;
    const int unit = blockIdx.x, lane = threadIdx.x;
    for (int e = lane; e < E * SZ; e += 64) sub[e] = 0.0;
    const int rl = lane & 15, vz = nu_vzero();
    int off[NP], oy[NP], oz[NP];
    bool ok[NP];
    double okf[NP];
#pragma unroll
    for (int ps = 0; ps < NP; ++ps) {
        const int j = lane + 64 * ps;
        ok[ps] = j < W * W;
        okf[ps] = ok[ps] ? 1.0 : 0.0;
        oy[ps] = ok[ps] ? j % W : 0;
        oz[ps] = ok[ps] ? j / W : 0;
        off[ps] = oz[ps] * SZ + oy[ps] * SY;
    }
    const int pbeg = unit_ptr[unit], pend = unit_ptr[unit + 1];
    double acc[NP][E];
#pragma unroll
    for (int ps = 0; ps < NP; ++ps)
#pragma unroll
        for (int k = 0; k < E; ++k) acc[ps][k] = 0.0;
    // adds the register rows into the subgrid row (by, bz) = (rw & 255, rw >> 8)
    auto flush = [&](int rw) {
        asm volatile("" ::: "memory");
        double *blk = sub + (rw >> 8) * SZ + (rw & 255) * SY;
#pragma unroll
        for (int ps = 0; ps < NP; ++ps)
            if (ok[ps]) {
                double *r = blk + off[ps];
#pragma unroll
                for (int k = 0; k < E; ++k) r[k] += acc[ps][k];
            }
        asm volatile("" ::: "memory");
#pragma unroll
        for (int ps = 0; ps < NP; ++ps)
#pragma unroll
            for (int k = 0; k < E; ++k) acc[ps][k] = 0.0;
    };
    NuPoint<NP> ring[D];
#pragma unroll
    for (int j = 0; j < D; ++j) nu_load<W, E, true>(ring[j], kval, qs, pbase, min(pbeg + j, pend - 1), rl, vz, oy, oz);
    int row = -1;
    for (int p0 = pbeg; p0 < pend; p0 += D) {
#pragma unroll
        for (int j = 0; j < D; ++j) {
            if (p0 + j < pend) {
                const NuPoint<NP> cur = ring[j];
                nu_load<W, E, true>(ring[j], kval, qs, pbase, min(p0 + j + D, pend - 1), rl, vz, oy, oz);
                const int rw = __builtin_amdgcn_readfirstlane(cur.pb) >> 8;
                if (rw != row) {
                    if (row >= 0) flush(row);
                    row = rw;
                }
#pragma unroll
                for (int ps = 0; ps < NP; ++ps)
                    dpp_row_axpy<E>(acc[ps], cur.ka, cur.kb, cur.q * cur.y[ps] * cur.z[ps] * okf[ps]);
            }
        }
    }
    if (row >= 0) flush(row);
    __syncthreads();
    constexpr int E2 = E * E, E3 = E2 * E;
    double *dst = scratch + (size_t)unit_slot[unit] * E3;
    for (int e = lane; e < E3; e += 64) dst[e] = sub[(e / E2) * SZ + ((e / E) % E) * SY + e % E];
}

// scratch[tile] += scratch[extra slots of the tile] (in unit order), for tiles split into
// several units.  Workgroup (chunk of 256 cells, listed tile).
__global__ __launch_bounds__(256) void k_nufft_extra_reduce(double *__restrict__ scratch, const int *__restrict__ extra_tile,
                                                            const int *__restrict__ extra_ptr, int n_tiles, int E3) {
    const int i = blockIdx.y, e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= E3) return;
    double v = scratch[(size_t)extra_tile[i] * E3 + e];
    for (int k = extra_ptr[i]; k < extra_ptr[i + 1]; ++k) v += scratch[(size_t)(n_tiles + k) * E3 + e];
    scratch[(size_t)extra_tile[i] * E3 + e] = v;
}

// grid[g] = sum over the tiles whose subgrid covers g (fixed order); tiles without points
// hold zeros.
__global__ __launch_bounds__(64) void k_nufft_gather(const double *__restrict__ scratch, const int *__restrict__ gp0,
                                                     const int *__restrict__ gt0, const int *__restrict__ gl0,
                                                     const int *__restrict__ gp1, const int *__restrict__ gt1,
                                                     const int *__restrict__ gl1, const int *__restrict__ gp2,
                                                     const int *__restrict__ gt2, const int *__restrict__ gl2, int n0, int n1,
                                                     int n2, int nt0, int nt1, int E, double *__restrict__ grid) {
    const int g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= n0 * n1 * n2) return;
    const int g0 = g % n0, g1 = (g / n0) % n1, g2 = g / (n0 * n1);
    const size_t E3 = (size_t)E * E * E;
    double v = 0;
    for (int a = gp2[g2]; a < gp2[g2 + 1]; ++a)
        for (int b = gp1[g1]; b < gp1[g1 + 1]; ++b) {
            const int tzy = gt2[a] * nt1 + gt1[b];
            const int lzy = gl2[a] * E + gl1[b];
            for (int c = gp0[g0]; c < gp0[g0 + 1]; ++c)
                v += scratch[(size_t)(tzy * nt0 + gt0[c]) * E3 + (size_t)lzy * E + gl0[c]];
        }
    grid[g] = v;
}

// out[a][k][b] = sum_l in[a][l][b] mat[k L + l] (complex matrix; real or complex input and
// output, the real output keeping the real part).  A lane owns one line (a, b) (b fastest, so
// the loads of a wavefront are contiguous when B > 1) and DFT_KC outputs k of it, grid y =
// the chunk of k: each input element read feeds DFT_KC complex multiply-adds, and the matrix
// entries are wave-uniform loads.  Each output is summed over l in order.
constexpr int DFT_KC = 8;

template <bool RIN, bool ROUT>
__global__ __launch_bounds__(256) void k_dft_axis(const void *__restrict__ in, void *__restrict__ out,
                                                  const double2 *__restrict__ mat, int A, int L, int K, int B) {
    const long col = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (col >= (long)A * B) return;
    const int b = (int)(col % B);
    const long a = col / B;
    const int k0 = blockIdx.y * DFT_KC;
    int row[DFT_KC];
#pragma unroll
    for (int j = 0; j < DFT_KC; ++j) row[j] = min(k0 + j, K - 1) * L;  // clamped rows are not stored
    double sr[DFT_KC], si[DFT_KC];
#pragma unroll
    for (int j = 0; j < DFT_KC; ++j) sr[j] = si[j] = 0.0;
    for (int l = 0; l < L; ++l) {
        const size_t ii = ((size_t)a * L + l) * B + b;
        if (RIN) {
            const double x = static_cast<const double *>(in)[ii];
#pragma unroll
            for (int j = 0; j < DFT_KC; ++j) {
                const double2 m = mat[row[j] + l];
                sr[j] = fma(x, m.x, sr[j]);
                si[j] = fma(x, m.y, si[j]);
            }
        } else {
            const double2 x = static_cast<const double2 *>(in)[ii];
#pragma unroll
            for (int j = 0; j < DFT_KC; ++j) {
                const double2 m = mat[row[j] + l];
                sr[j] = fma(x.x, m.x, fma(-x.y, m.y, sr[j]));
                si[j] = fma(x.x, m.y, fma(x.y, m.x, si[j]));
            }
        }
    }
#pragma unroll
    for (int j = 0; j < DFT_KC; ++j) {
        if (k0 + j >= K) break;
        const size_t o = ((size_t)a * K + k0 + j) * B + b;
        if (ROUT) static_cast<double *>(out)[o] = sr[j];
        else static_cast<double2 *>(out)[o] = make_double2(sr[j], si[j]);
    }
}

// C[pos[i]] = cw[i] B[pos[i]] for the listed modes (the other entries of C stay zero).
__global__ void k_nufft_coef(const double2 *__restrict__ Bbox, const int *__restrict__ pos, const double *__restrict__ cw,
                             int n_modes, double2 *__restrict__ Cbox) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n_modes) return;
    const double2 v = Bbox[pos[i]];
    Cbox[pos[i]] = make_double2(cw[i] * v.x, cw[i] * v.y);
}

// Row stride of the interpolation kernel's partial sums (odd, so that lane i reading row i
// spreads over the banks), and points per partial-sum batch.
constexpr int NU_PS = 65, NU_IB = 32;

// One wavefront per work unit: the tile subgrid (periodic wrap of the grid) is staged in
// LDS; for each subgrid row (by, bz) the lanes load their rows into registers and, per point,
// form sum_x phi_x row[x] phi_y phi_z over their offsets (dy, dz); the 64 lane partials of
// each point are added in lane order.  far[i] = the interpolated value at the point in plan
// position i.
template <int W, int E>
__global__ __launch_bounds__(64) void k_nufft_interp(const double *__restrict__ grid, const int *__restrict__ unit_ptr,
                                                     const int *__restrict__ unit_tile, const double *__restrict__ kval,
                                                     const int *__restrict__ pbase, int n0, int n1, int n2, int nt0, int nt1,
                                                     int T, int lo, int SY, int SZ, double *__restrict__ far) {
    using C = NufftCfg<W, E>;
    constexpr int NP = C::NP, D = C::D;
    extern __shared__ double nu_lds[];
    const int unit = blockIdx.x, lane = threadIdx.x;
    double *sub = nu_lds, *part = nu_lds + E * SZ;
    int *wrap = reinterpret_cast<int *>(part + NU_IB * NU_PS);  // 3 E grid indices
    const int rl = lane & 15, vz = nu_vzero();
    int off[NP], oy[NP], oz[NP];
    double okf[NP];
#pragma unroll
    for (int ps = 0; ps < NP; ++ps) {
        const int j = lane + 64 * ps;
        const bool ok = j < W * W;
        okf[ps] = ok ? 1.0 : 0.0;
        oy[ps] = ok ? j % W : 0;
        oz[ps] = ok ? j / W : 0;
        off[ps] = oz[ps] * SZ + oy[ps] * SY;
    }
    const int pbeg = unit_ptr[unit], pend = unit_ptr[unit + 1];
    NuPoint<NP> ring[D];
#pragma unroll
    for (int j = 0; j < D; ++j) nu_load<W, E, false>(ring[j], kval, nullptr, pbase, min(pbeg + j, pend - 1), rl, vz, oy, oz);
    const int tile = unit_tile[unit];
    const int org[3] = {T * (tile % nt0) + lo, T * ((tile / nt0) % nt1) + lo, T * (tile / (nt0 * nt1)) + lo};
    const int nn[3] = {n0, n1, n2};
#pragma unroll
    for (int d = 0; d < 3; ++d)
        if (lane < E) wrap[d * E + lane] = ((org[d] + lane) % nn[d] + nn[d]) % nn[d];
    __syncthreads();
    {
        constexpr int E2 = E * E, E3 = E2 * E;
        for (int e0 = 0; e0 < E3; e0 += 256) {
            double v[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int e = min(e0 + 64 * u + lane, E3 - 1);
                v[u] = grid[((size_t)wrap[2 * E + e / E2] * n1 + wrap[E + (e / E) % E]) * n0 + wrap[e % E]];
            }
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int e = e0 + 64 * u + lane;
                if (e < E3) sub[(e / E2) * SZ + ((e / E) % E) * SY + e % E] = v[u];
            }
        }
    }
    __syncthreads();
    double col[NP][E];
    int row = -1, bstart = pbeg, nb = 0;
    // far for the nb points from bstart: lane i adds row i of the partial sums
    auto reduce = [&](int n_pts) {
        asm volatile("" ::: "memory");
        if (lane < n_pts) {
            double s = 0;
            for (int l = 0; l < 64; ++l) s += part[lane * NU_PS + l];
            far[bstart + lane] = s;
        }
        asm volatile("" ::: "memory");
    };
    for (int p0 = pbeg; p0 < pend; p0 += D) {
#pragma unroll
        for (int j = 0; j < D; ++j) {
            if (p0 + j < pend) {
                const NuPoint<NP> cur = ring[j];
                nu_load<W, E, false>(ring[j], kval, nullptr, pbase, min(p0 + j + D, pend - 1), rl, vz, oy, oz);
                const int rw = __builtin_amdgcn_readfirstlane(cur.pb) >> 8;
                if (rw != row) {
                    row = rw;
                    const double *blk = sub + (row >> 8) * SZ + (row & 255) * SY;
#pragma unroll
                    for (int ps = 0; ps < NP; ++ps)
#pragma unroll
                        for (int k = 0; k < E; ++k) col[ps][k] = blk[off[ps] + k];
                }
                double acc = 0;
#pragma unroll
                for (int ps = 0; ps < NP; ++ps) {
                    double s0 = 0, s1 = 0;
                    dpp_row_dot<E>(s0, s1, cur.ka, cur.kb, col[ps]);
                    acc = fma(s0 + s1, cur.y[ps] * cur.z[ps] * okf[ps], acc);
                }
                part[nb * NU_PS + lane] = acc;
                if (++nb == NU_IB) {
                    reduce(NU_IB);
                    bstart += NU_IB;
                    nb = 0;
                }
            }
        }
    }
    reduce(nb);
}

// ------------------------------------------------------------------ quasi-periodic far field
// psi(x_u) = e^{i b.x_u} sum_m w_m S(m) e^{i m.theta_u},  S(m) = sum_l q_l e^{-i b.x_l}
// e^{-i m.theta_l}, over the full mode box m = (i, j, k) - (ms/2, mt/2, mu/2), index
// i + ms (j + mt k); w_m = 0 outside the window (cpp/src/dmk/pbc.cpp:249-355).  FP64.
// Sp[y][m]: partial structure factors of the points of workgroup column y.  Per tile of tp
// points the per-axis factors e^{-i m_d theta_d} are tabulated in LDS by recurrence
// (tp (ms + mt + mu + 2) complex values); a thread owns QP_CHUNK consecutive i of one (j, k)
// line and walks them by multiplying with e^{-i theta_1}, so a (point, mode) pair costs one
// complex multiply-add.
//
// For FP32 trees, whose values are rounded to FP32 after this FP64 sum: k_ff_* add in another
// order, and a value in about 2e6 falls on the other side of its rounding.  evaluate_complex()
// at 6 digits, FP32: N = 1e3 1100 us with the walks of one thread (reduction, evaluation) one
// load after another, 214 with them split as below; 3e4 1755 / 470; 1e5 2370 / 1050 (k_ff_*: 180,
// 408, 670).  Bound by FP64 vector issue: k_qp_structure 520 us beside the chain at N = 1e5.
constexpr int QP_CHUNK = 8;
__global__ __launch_bounds__(256) void k_qp_structure(const double *__restrict__ theta, const double *__restrict__ bx,
                                                       const double *__restrict__ q, int n, int ms, int mt, int mu, int tp,
                                                       double2 *__restrict__ Sp) {
    extern __shared__ double2 qp_lds[];
    double2 *E1 = qp_lds, *E2 = E1 + tp * ms, *E3 = E2 + tp * mt, *Q = E3 + tp * mu, *Est = Q + tp;
    const int M = ms * mt * mu, nci = (ms + QP_CHUNK - 1) / QP_CHUNK;
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    const bool active = c < nci * mt * mu;
    const int i0 = active ? QP_CHUNK * (c % nci) : 0, j = active ? (c / nci) % mt : 0, k = active ? c / (nci * mt) : 0;
    double2 acc[QP_CHUNK];
#pragma unroll
    for (int r = 0; r < QP_CHUNK; ++r) acc[r] = make_double2(0, 0);
    for (int p0 = blockIdx.y * tp; p0 < n; p0 += gridDim.y * tp) {
        __syncthreads();
        for (int t = threadIdx.x; t < tp * 4; t += blockDim.x) {
            const int pp = t % tp, ax = t / tp, gp = p0 + pp;
            if (ax == 3) {  // q e^{-i b.x}
                double sn = 0, cs = 0;
                if (gp < n) {
                    sincos(-bx[gp], &sn, &cs);
                    sn *= q[gp];
                    cs *= q[gp];
                }
                Q[pp] = make_double2(cs, sn);
                continue;
            }
            const int cnt = ax == 0 ? ms : (ax == 1 ? mt : mu);
            double2 *row = (ax == 0 ? E1 : (ax == 1 ? E2 : E3)) + pp * cnt;
            const double th = gp < n ? theta[3 * (size_t)gp + ax] : 0.0;
            double s1, c1, sl, cl;
            sincos(th, &s1, &c1);
            sincos(th * (cnt / 2), &sl, &cl);
            const double2 step = make_double2(c1, -s1);  // e^{-i th}
            if (ax == 0) Est[pp] = step;
            double2 cur = make_double2(cl, sl);  // e^{-i (-(cnt/2)) th}
            for (int mm = 0; mm < cnt; ++mm) {
                row[mm] = cur;
                cur = cmul(cur, step);
            }
        }
        __syncthreads();
        if (active) {
            const int np = min(tp, n - p0);
            for (int pp = 0; pp < np; ++pp) {
                const double2 st = Est[pp];
                double2 cur = cmul(cmul(cmul(E1[pp * ms + i0], E2[pp * mt + j]), E3[pp * mu + k]), Q[pp]);
#pragma unroll
                for (int r = 0; r < QP_CHUNK; ++r) {
                    acc[r].x += cur.x;
                    acc[r].y += cur.y;
                    cur = cmul(cur, st);
                }
            }
        }
    }
    if (active) {
        const int m0 = i0 + ms * (j + mt * k);
#pragma unroll
        for (int r = 0; r < QP_CHUNK; ++r)
            if (i0 + r < ms) Sp[(size_t)blockIdx.y * M + m0 + r] = acc[r];
    }
}

// S[m] = w[m] sum_y Sp[y][m], partials added in column order, QP_AHEAD loads in flight (N = 3e4 at
// 3 digits, 1876 columns: 584 us one at a time, 60 with 32).
constexpr int QP_AHEAD = 32;
__global__ __launch_bounds__(64) void k_qp_reduce(const double2 *__restrict__ Sp, int nblk, const double *__restrict__ w,
                                                  int M, double2 *__restrict__ S) {
    const int m = blockIdx.x * blockDim.x + threadIdx.x;
    if (m >= M) return;
    double2 a = make_double2(0, 0);
    int b = 0;
    for (; b + QP_AHEAD <= nblk; b += QP_AHEAD) {
        double2 v[QP_AHEAD];
#pragma unroll
        for (int i = 0; i < QP_AHEAD; ++i) v[i] = Sp[(size_t)(b + i) * M + m];
#pragma unroll
        for (int i = 0; i < QP_AHEAD; ++i) {
            a.x += v[i].x;
            a.y += v[i].y;
        }
    }
    for (; b < nblk; ++b) {
        const double2 v = Sp[(size_t)b * M + m];
        a.x += v.x;
        a.y += v.y;
    }
    S[m] = make_double2(a.x * w[m], a.y * w[m]);
}

// far[u] = psi(x_u), 64 points per workgroup.  The i axis is taken in chunks of QP_CHUNK: the
// chunk's factors e^{i m_1 theta_1} sit in registers and serve every (j, k) line, whose factors
// follow recurrences in e^{i theta_2}, e^{i theta_3}; the weighted structure factors are read at
// wave-uniform addresses.  The QP_EW waves take (chunk, k) planes in turn, and wave 0 adds their
// sums in plane order, as one wave does that walks all planes (718 us at N = 1e5, this 350 beside
// the chain).
constexpr int QP_EW = 8;
__global__ __launch_bounds__(64 * QP_EW) void k_qp_eval(const double *__restrict__ theta, const double *__restrict__ bx,
                                                        int n, int ms, int mt, int mu, const double2 *__restrict__ S,
                                                        double2 *__restrict__ far) {
    __shared__ double2 part[2][QP_EW][64];
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int u = blockIdx.x * 64 + lane, uc = min(u, n - 1);
    double2 st[3], e[3];
    const int cnt[3] = {ms, mt, mu};
    for (int d = 0; d < 3; ++d) {
        const double th = theta[3 * (size_t)uc + d];
        double sn, cs;
        sincos(th, &sn, &cs);
        e[d] = make_double2(cs, sn);  // e^{i th}
        sincos(-th * (cnt[d] / 2), &sn, &cs);
        st[d] = make_double2(cs, sn);  // e^{i (-(cnt/2)) th}
    }
    const int planes = (ms + QP_CHUNK - 1) / QP_CHUNK * mu;
    int chunk = -1, kc = 0;  // the chunk in c1, the plane of c3
    double2 acc = make_double2(0, 0), c1next = st[0], c3 = st[2], c1[QP_CHUNK];
    for (int p0 = 0, buf = 0; p0 < planes; p0 += QP_EW, buf ^= 1) {
        const int p = p0 + w, c = p / mu, k = p - c * mu, i0 = c * QP_CHUNK;
        if (p < planes) {
            while (chunk < c) {
#pragma unroll
                for (int r = 0; r < QP_CHUNK; ++r) {
                    c1[r] = c1next;
                    c1next = cmul(c1next, e[0]);
                }
                ++chunk;
                kc = 0;
                c3 = st[2];
            }
            for (; kc < k; ++kc) c3 = cmul(c3, e[2]);
            const int nr = min(QP_CHUNK, ms - i0);
            double2 acc2 = make_double2(0, 0), c2 = st[1];
            for (int j = 0; j < mt; ++j) {
                const double2 *row = S + ((size_t)k * mt + j) * ms + i0;
                double2 l = make_double2(0, 0);
#pragma unroll
                for (int r = 0; r < QP_CHUNK; ++r) {
                    if (r < nr) {
                        const double2 v = row[r];
                        l.x = fma(v.x, c1[r].x, fma(-v.y, c1[r].y, l.x));
                        l.y = fma(v.x, c1[r].y, fma(v.y, c1[r].x, l.y));
                    }
                }
                const double2 t2 = cmul(l, c2);
                acc2.x += t2.x;
                acc2.y += t2.y;
                c2 = cmul(c2, e[1]);
            }
            part[buf][w][lane] = cmul(acc2, c3);
        }
        __syncthreads();
        // (the other buffer is written meanwhile, this one again only after the next barrier)
        if (w == 0)
            for (int i = 0; i < min(QP_EW, planes - p0); ++i) {
                acc.x += part[buf][i][lane].x;
                acc.y += part[buf][i][lane].y;
            }
    }
    if (w == 0 && u < n) {
        double sn, cs;
        sincos(bx[u], &sn, &cs);
        far[u] = cmul(acc, make_double2(cs, sn));
    }
}

}  // namespace pdmk::gpu
