// mck_mfma.inc.h - backward evaluation through element spectra and the matrix cores.
//
// The backward strain of a (point, receiver) pair is a linear map of the nodal traces of
// one backward element: B_c(t) = sum_j W_c,j u_j(t) over the element's traces j (the
// variables the receiver component reads x 25 GLL nodes; the weights hold the strain
// operator, the Lagrange interpolation at (xi, eta) and the azimuthal factors,
// readfields.f90:1359-1465, sem_derivatives.f90, spectral_basis.f90:181-314).  Taper, zero
// padding and the real FFT are linear too (fft.f90:375-413, 546-601), so
//     B_c(k) = sum_j W_c,j U_j(k),    U_j = rfft(taper . u_j)
// The nodal spectra U of every backward element a launch touches are computed once
// (k_elem_spectra); the pairs of an element then form their
// spectra as one matrix product [bins x traces] x [traces x pairs] on the matrix cores
// (fp32 operands as split fp16 products), fused with the frequency-domain contraction of
// k_bwd_eval: base kernels per bin (kernel.f90:514-570) against the forward spectra of
// the pair's point, the filtered window integrals sum_k Re(bk_k H_k) accumulated in FP64
// (kernel.f90:410-510, 946-1020), and the physical kernels (kernel.f90:665-832).
//
// Pairs arrive sorted by (element, receiver); a run is the pairs of one element.
#pragma once

namespace mck {


// Work tables of element- and receiver-sorted pair keys (element * R + receiver):
// element runs (the elements whose spectra a launch needs) and groups of at most 16
// consecutive pairs with one key (one workgroup of k_bwd_mfma each).
// flags: eflag[i] = a new element starts at i, kflag[i] = a new key starts at i
__global__ void k_run_flags(int n, const int *keys, int R, int *eflag, int *kflag)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    eflag[i] = (i == 0 || keys[i] / R != keys[i - 1] / R) ? 1 : 0;
    kflag[i] = (i == 0 || keys[i] != keys[i - 1]) ? 1 : 0;
}

// from the inclusive scans of the flags (epos, kpos): element runs erun_first[u] (with
// erun_first[nerun] = n), erun_elem[u], *nerun; first item of every key run krun_first[v];
// gflag[i] = a group starts at i (every 16th item of a key run)
__global__ void k_run_table(int n, const int *keys, int R, const int *eflag, const int *epos, const int *kflag,
                            const int *kpos, int *erun_first, int *erun_elem, int *nerun, int *krun_first)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    if (eflag[i]) {
        const int u = epos[i] - 1;
        erun_first[u] = i;
        erun_elem[u] = keys[i] / R;
    }
    if (kflag[i]) krun_first[kpos[i] - 1] = i;
    if (i == n - 1) {
        *nerun = epos[i];
        erun_first[epos[i]] = n;
    }
}

__global__ void k_group_flags(int n, const int *kpos, const int *krun_first, int *gflag)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    gflag[i] = ((i - krun_first[kpos[i] - 1]) & 15) == 0 ? 1 : 0;
}

// groups from the inclusive scan of gflag: group_first[g] (with group_first[ngroups] = n),
// the element run of the group, the first group of every element run (an element run
// starts a group; erun_group_first[nerun] = ngroups), *ngroups
__global__ void k_group_table(int n, const int *gflag, const int *gpos, const int *eflag, const int *epos,
                              int *group_first, int *group_erun, int *erun_group_first, int *ngroups)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    if (gflag[i]) {
        const int g = gpos[i] - 1;
        group_first[g] = i;
        group_erun[g] = epos[i] - 1;
        if (eflag[i]) erun_group_first[epos[i] - 1] = g;
    }
    if (i == n - 1) {
        *ngroups = gpos[i];
        group_first[gpos[i]] = n;
        erun_group_first[epos[i]] = gpos[i];
    }
}

// ------------------------------------------------------------------------------------
// k_elem_spectra: the tapered real spectra (x dt) of the J = nvar_bwd x 25 nodal traces of
// the elements of runs u0 .. u0 + gridDim.x - 1, U[u - u0][tile][j][16 bins] (tile_at; zero
// beyond bin M).  Computed in double precision and rounded once: the spectra of an
// element serve all of its pairs.
//
// A trace's FFT (z[n] = x[2n] + i x[2n + 1], length M = 512 .. 4096, its upper half zero)
// runs on M / 16 threads with 16 values each in registers: radix 16, 16 and M / 256
// (Stockham order), so that it crosses LDS twice instead of once per radix-4 pass, with
// twiddles kept in registers from trace to trace; the real spectrum's bins k and M - k
// come from one pair of values.  A workgroup holds G traces at a time; blockIdx.y: a share
// of the traces, so that few elements still fill the chip.
// Bound: HBM (25 KB per trace of 2048 samples) and LDS about equally.  3,186 elements of
// nt 2048 (3.9 GB): 2.73 ms with radix-4 passes through two LDS buffers and twiddles from
// memory, 1.25 ms (3.1 TB/s; a large copy reaches 4.9); 895 elements of nt 4096 2.76 ->
// 0.78 ms; 15 elements of nt 1024 184 -> 22 us (their traces spread over workgroups).
// ------------------------------------------------------------------------------------
template <int M>
struct ElemFft {
    static constexpr int T = M / 16;                       // threads of a trace
    static constexpr int BLK = T < 64 ? 64 : T;            // threads of a workgroup
    static constexpr int G = BLK / T;                      // traces at a time
    static constexpr int LDS = M + M / 16 + 1;             // padded values of a trace, and z[0] once more
    static constexpr int R = M / 256;                      // last radix
    static constexpr size_t smem = (size_t)G * LDS * sizeof(double2);
};

// LDS slot of value i: one padding slot after every 16 (T is a multiple of 16: slots of
// i + T q are a constant apart)
__device__ __forceinline__ int elem_slot(int i) { return i + (i >> 4); }
__device__ __forceinline__ double2 dadd(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ double2 dsub(double2 a, double2 b) { return make_double2(a.x - b.x, a.y - b.y); }

// a (cos, sin) constant: a e^{-i phi}
__device__ __forceinline__ double2 drot(double2 a, double c, double s)
{
#pragma clang fp contract(fast)
    return make_double2(a.x * c + a.y * s, a.y * c - a.x * s);
}
__device__ __forceinline__ double2 dmul(double2 a, double2 b)
{
#pragma clang fp contract(fast)
    return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}

// 4-point DFT (e^{-2 pi i / 4}); HALF: c and d are zero
template <bool HALF>
__device__ __forceinline__ void dft4(double2 &a, double2 &b, double2 &c, double2 &d)
{
    const double2 s0 = HALF ? a : dadd(a, c), d0 = HALF ? a : dsub(a, c);
    const double2 s1 = HALF ? b : dadd(b, d), d1 = HALF ? b : dsub(b, d);
    a = dadd(s0, s1);
    b = make_double2(d0.x + d1.y, d0.y - d1.x);
    c = dsub(s0, s1);
    d = make_double2(d0.x - d1.y, d0.y + d1.x);
}

// R-point DFT of v[0..R) in place; output r is v[dft_at<R>(r)].  HALF: the upper half of
// the inputs is zero (R 16)
template <int R>
__host__ __device__ constexpr int dft_at(int r) { return R == 16 ? (r >> 2) + 4 * (r & 3) : (R == 8 ? (r >> 2) + 2 * (r & 3) : r); }

template <int R, bool HALF = false>
__device__ __forceinline__ void dft(double2 *v)
{
    constexpr double c8 = 0.70710678118654752440, c16 = 0.92387953251128675613, s16 = 0.38268343236508977173;
    if constexpr (R == 2) {
        const double2 a = v[0], b = v[1];
        v[0] = dadd(a, b);
        v[1] = dsub(a, b);
    } else if constexpr (R == 4) {
        dft4<false>(v[0], v[1], v[2], v[3]);
    } else if constexpr (R == 8) {
        dft4<false>(v[0], v[2], v[4], v[6]);
        dft4<false>(v[1], v[3], v[5], v[7]);
        v[3] = drot(v[3], c8, c8);
        v[5] = make_double2(v[5].y, -v[5].x);
        v[7] = drot(v[7], -c8, c8);
#pragma unroll
        for (int r = 0; r < 8; r += 2) {
            const double2 a = v[r], b = v[r + 1];
            v[r] = dadd(a, b);
            v[r + 1] = dsub(a, b);
        }
    } else {
#pragma unroll
        for (int q = 0; q < 4; ++q) dft4<HALF>(v[q], v[q + 4], v[q + 8], v[q + 12]);
        v[5] = drot(v[5], c16, s16);
        v[6] = drot(v[6], c8, c8);
        v[7] = drot(v[7], s16, c16);
        v[9] = drot(v[9], c8, c8);
        v[10] = make_double2(v[10].y, -v[10].x);
        v[11] = drot(v[11], -c8, c8);
        v[13] = drot(v[13], s16, c16);
        v[14] = drot(v[14], -c8, c8);
        v[15] = drot(v[15], -c16, -s16);
#pragma unroll
        for (int q = 0; q < 16; q += 4) dft4<false>(v[q], v[q + 1], v[q + 2], v[q + 3]);
    }
}

// v[q] *= w^q, q = 1 .. R - 1, from w^1, w^2, w^4, w^8
template <int R>
__device__ __forceinline__ void elem_twiddle(double2 *v, const double2 *w)
{
    v[1] = dmul(v[1], w[0]);
    if constexpr (R >= 4) {
        const double2 w3 = dmul(w[0], w[1]);
        v[2] = dmul(v[2], w[1]);
        v[3] = dmul(v[3], w3);
        if constexpr (R >= 8) {
            const double2 w5 = dmul(w[0], w[2]), w6 = dmul(w[1], w[2]), w7 = dmul(w3, w[2]);
            v[4] = dmul(v[4], w[2]);
            v[5] = dmul(v[5], w5);
            v[6] = dmul(v[6], w6);
            v[7] = dmul(v[7], w7);
            if constexpr (R >= 16) {
                v[8] = dmul(v[8], w[3]);
                v[9] = dmul(v[9], dmul(w[0], w[3]));
                v[10] = dmul(v[10], dmul(w[1], w[3]));
                v[11] = dmul(v[11], dmul(w3, w[3]));
                v[12] = dmul(v[12], dmul(w[2], w[3]));
                v[13] = dmul(v[13], dmul(w5, w[3]));
                v[14] = dmul(v[14], dmul(w6, w[3]));
                v[15] = dmul(v[15], dmul(w7, w[3]));
            }
        }
    }
}

template <int M>
__global__ __launch_bounds__(ElemFft<M>::BLK, 2) void k_elem_spectra(DevDb db, PathConf pc, int u0, int nrun,
                                                                     const int *run_elem,
                                                                     const double2 *__restrict__ twd, float2 *U)
{
    using E = ElemFft<M>;
    constexpr int T = E::T, R = E::R, NB = 16 / R, N = 2 * M, lq = 30 - __builtin_clz(M);    // 2^lq = N / 4
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const int u = u0 + (int)blockIdx.x;
    if (u >= nrun) return;
    const float *ue = elem_u(db, run_elem[u]);
    if (!ue) return;
    const int g = (int)threadIdx.x / T, t = (int)threadIdx.x % T;
    double2 *z = reinterpret_cast<double2 *>(smem_raw) + g * E::LDS;
    const int J = pc.nvar_bwd * 25, nt = pc.nt;
    const bool pairs = (nt & 1) == 0;                      // sample pairs aligned
    // twiddle powers 1, 2, 4, 8 of the second pass (w_256^(t % 16)) and of the NB last
    // butterflies (w_M^j, j = t + T b)
    double2 wb[4], wc[NB][4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        wb[i] = twiddle_d(twd, ((t & 15) << i) * (N / 256), lq);
#pragma unroll
        for (int b = 0; b < NB; ++b)
            if ((1 << i) < R) wc[b][i] = twiddle_d(twd, ((t + T * b) << i) * 2, lq);
    }
    float2 *Uu = U + (size_t)(u - u0) * J * pc.ustride;
    // this block's share of the traces, G at a time
    const int ng = (J + E::G - 1) / E::G;
    const int i0 = (int)blockIdx.y * ng / (int)gridDim.y, i1 = ((int)blockIdx.y + 1) * ng / (int)gridDim.y;
    float nx[16];
    auto load = [&](int i) {
        const int j = min(i * E::G + g, J - 1);
        const int src = (pc.bwd_vars[j / 25] * 25 + j % 25) * nt;
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const int n = 2 * (t + T * q);
            nx[2 * q] = nx[2 * q + 1] = 0.0f;
            if (pairs) {
                if (n < nt) {
                    const float2 v = gload2(ue, src + n);
                    nx[2 * q] = v.x;
                    nx[2 * q + 1] = v.y;
                }
            } else {
                if (n < nt) nx[2 * q] = gload1(ue, src + n);
                if (n + 1 < nt) nx[2 * q + 1] = gload1(ue, src + n + 1);
            }
        }
    };
    if (i0 < i1) load(i0);
    for (int i = i0; i < i1; ++i) {
        double2 v[16];
        // (the products of the twiddle powers and the last pass's twiddles are formed or loaded
        // for every trace: kept across the loop they would not fit the registers)
        int k0 = t;
        asm volatile("" : "+v"(k0), "+v"(wb[0].x), "+v"(wb[1].x), "+v"(wb[2].x), "+v"(wb[3].x));
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int p = 0; p < 4; ++p)
                if ((1 << p) < R) asm volatile("" : "+v"(wc[b][p].x));
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            v[q] = make_double2((double)nx[2 * q], (double)nx[2 * q + 1]);
            const int n = 2 * (t + T * q);
            if (n < pc.ntaper || n + 1 >= nt - pc.ntaper) {
                float tp[2];
                taper_factors(n, nt, pc, tp);
                v[q].x *= tp[0];
                v[q].y *= tp[1];
            }
            v[q + 8] = make_double2(0.0, 0.0);
        }
        if (i + 1 < i1) load(i + 1);
        dft<16, true>(v);
#pragma unroll
        for (int r = 0; r < 16; ++r) z[17 * t + r] = v[dft_at<16>(r)];
        __syncthreads();
#pragma unroll
        for (int q = 0; q < 16; ++q) v[q] = z[elem_slot(t) + q * (T + T / 16)];
        __syncthreads();
        elem_twiddle<16>(v, wb);
        dft<16>(v);
#pragma unroll
        for (int r = 0; r < 16; ++r) z[(t >> 4) * 272 + (t & 15) + 17 * r] = v[dft_at<16>(r)];
        __syncthreads();
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int q = 0; q < R; ++q) v[b * R + q] = z[elem_slot(t) + b * (T + T / 16) + 272 * q];
        __syncthreads();
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            elem_twiddle<R>(v + b * R, wc[b]);
            dft<R>(v + b * R);
#pragma unroll
            for (int r = 0; r < R; ++r) z[elem_slot(t) + b * (T + T / 16) + 272 * r] = v[b * R + dft_at<R>(r)];
        }
        if (t == 0) z[E::LDS - 1] = v[dft_at<R>(0)];
        __syncthreads();
        // X_k = E_k + w_N^k O_k and X_(M - k) = conj(E_k - w_N^k O_k)
        const int j = i * E::G + g;
        if (j < J) {
            // (T is a multiple of 16: the bins t + T q and M - t - T q are T J apart)
            float2 *dk = Uu + tile_at(J, j, t), *dm = Uu + tile_at(J, j, M - t);
            const double dt = pc.dt;
#pragma unroll
            for (int q = 0; q < 8; ++q) {
#pragma clang fp contract(fast)
                const double2 zk = z[elem_slot(t) + q * (T + T / 16)], zm = z[elem_slot(M - t) - q * (T + T / 16)];
                const double2 w = twd[k0 + T * q];
                const double ex = 0.5 * (zk.x + zm.x), ey = 0.5 * (zk.y - zm.y);
                const double ox = 0.5 * (zk.y + zm.y), oy = 0.5 * (zm.x - zk.x);
                const double px = w.x * ox - w.y * oy, py = w.x * oy + w.y * ox;
                dk[(size_t)q * T * J] = make_float2((float)((ex + px) * dt), (float)((ey + py) * dt));
                dm[-(ptrdiff_t)q * T * J] = make_float2((float)((ex - px) * dt), (float)((py - ey) * dt));
            }
            if (t == 0) {
                const double2 zh = z[elem_slot(M / 2)];
                Uu[tile_at(J, j, M / 2)] = make_float2((float)(zh.x * dt), (float)(-zh.y * dt));
            }
            for (int k = M + 1 + t; k < pc.ustride; k += T) Uu[tile_at(J, j, k)] = make_float2(0.0f, 0.0f);
        }
        __syncthreads();
    }
}

// the same for traces of at most 256 samples (M = 2 .. 256): one workgroup per element run,
// one sample per thread
__global__ __launch_bounds__(kStrainThreads) void k_elem_spectra_short(DevDb db, PathConf pc, int u0, int nrun,
                                                                       const int *run_elem, const double2 *twd,
                                                                       float2 *U)
{
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const int M = pc.M;
    double2 *bufA = reinterpret_cast<double2 *>(smem_raw);
    double2 *bufB = bufA + M;
    const int u = u0 + (int)blockIdx.x;
    if (u >= nrun) return;
    const float *ue = elem_u(db, run_elem[u]);
    if (!ue) return;
    const int tid = threadIdx.x, nt = pc.nt;
    const size_t blk = (size_t)25 * nt;
    float tap[1];
    taper_factors(tid, nt, pc, tap);
    const int J = pc.nvar_bwd * 25;
    float2 *Uu = U + (size_t)(u - u0) * J * pc.ustride;
    for (int j = 0; j < J; ++j) {
        const float *src = ue + (size_t)pc.bwd_vars[j / 25] * blk + (size_t)(j % 25) * nt;
        const double x = tid < nt ? (double)src[tid] * tap[0] : 0.0;
        const double2 *Z = lds_fft_d(x, tid, nt, M, bufA, bufB, twd);
        for (int k = tid; k < pc.ustride; k += kStrainThreads)
            Uu[tile_at(J, j, k)] = k <= M ? rfft_bin_d(Z, k, M, twd, pc.dt) : make_float2(0.0f, 0.0f);
        __syncthreads();
    }
}

constexpr int kMfmaPairs = 16;         // pairs of one wave (the matrix-core columns)
constexpr int kMfmaWaves = 4;          // waves of a workgroup of k_bwd_mfma (one group)

// The contraction U W of the element spectra with the pair weights on the fp16 matrix
// cores (v_mfma_f32_16x16x32_f16): every fp32 operand x is split into x_hi = fp16(x) and
// x_lo = fp16(x - x_hi), 22 of its 24 significant bits, and U W = U_hi W_hi + U_hi W_lo +
// U_lo W_hi (fp16 products are exact in fp32; the dropped U_lo W_lo is below 2^-22 of a
// product).  The operands are scaled by powers of two into fp16's range first (W per pair,
// U per tile of 16 bins, to below 2^14) and the base kernels scaled back.  K: one block of
// 32 per variable, its 25 nodal traces (8 per lane) and 7 zeros, so that a component skips
// the variables its strain does not contain.
typedef _Float16 v8h __attribute__((ext_vector_type(8)));

constexpr int mfma_ks(int nvb) { return 8 * nvb; }     // element spectra per lane

// whether carried component c contains variable v (sem_derivatives.f90:281-649): monopole
// fields (u_s, u_z: ss, pp, zz, sz), dipole fields (u_s, u_p, u_z: the Voigt six), traces
__host__ __device__ constexpr bool mfma_has(int ndb, int v, int c)
{
    if (ndb == 1) return true;
    if (ndb == 4) return v == 0 ? c != 2 : c >= 2;
    return v == 0 ? (c != 2 && c != 3) : (v == 1 ? (c == 1 || c == 3 || c == 5) : (c >= 2 && c <= 4));
}
// index of (v, c) among the blocks a group's weights are stored in, and their number
__host__ __device__ constexpr int mfma_wblock(int ndb, int v, int c)
{
    int n = 0;
    for (int i = 0; i < v * ndb + c; ++i) n += mfma_has(ndb, i / ndb, i % ndb) ? 1 : 0;
    return n;
}
__host__ __device__ constexpr int mfma_nblock(int ndb, int nvb) { return mfma_wblock(ndb, nvb, 0); }

// the largest of a non-negative value over the wave (all 64 lanes active): within each
// row of 16 lanes by DPP (lane swaps 1 and 2, rotations by 4 and 8), then across the 4
// rows on the bit patterns (non-negative floats order as unsigned integers)
__device__ __forceinline__ float mfma_wave_max(float x)
{
    unsigned v = __builtin_bit_cast(unsigned, x), o;
    o = (unsigned)__builtin_amdgcn_mov_dpp((int)v, 0xB1, 0xF, 0xF, true);
    v = v > o ? v : o;
    o = (unsigned)__builtin_amdgcn_mov_dpp((int)v, 0x4E, 0xF, 0xF, true);
    v = v > o ? v : o;
    o = (unsigned)__builtin_amdgcn_mov_dpp((int)v, 0x124, 0xF, 0xF, true);
    v = v > o ? v : o;
    o = (unsigned)__builtin_amdgcn_mov_dpp((int)v, 0x128, 0xF, 0xF, true);
    v = v > o ? v : o;
    const unsigned r0 = (unsigned)__builtin_amdgcn_readlane((int)v, 0), r1 = (unsigned)__builtin_amdgcn_readlane((int)v, 16);
    const unsigned r2 = (unsigned)__builtin_amdgcn_readlane((int)v, 32), r3 = (unsigned)__builtin_amdgcn_readlane((int)v, 48);
    const unsigned m = r0 > r1 ? r0 : r1, n = r2 > r3 ? r2 : r3;
    return __builtin_bit_cast(float, m > n ? m : n);
}

// (No instruction is written in asm here: the compiler keeps the wait states that matrix and
// DPP instructions need around the vector instructions it forms itself, not around asm.)

// max(m, |a|, |b|) in one instruction (the IEEE maximum: fmaxf would quiet NaNs first)
__device__ __forceinline__ float mfma_max3(float m, float a, float b)
{
    return __builtin_elementwise_maximum(__builtin_elementwise_maximum(m, fabsf(a)), fabsf(b));
}

// x, y (scaled into fp16's range) = hi + lo to 22 bits, as packed halves: fp16 conversion in
// pairs and the remainders by one mixed-precision FMA each (exact).  neg: -1 whose value
// the compiler does not see (mfma_neg_one): x - (float)h would take two instructions.
typedef _Float16 v2h __attribute__((ext_vector_type(2)));
__device__ __forceinline__ float mfma_neg_one()
{
    float neg = -1.0f;
    asm("" : "+s"(neg));
    return neg;
}
__device__ __forceinline__ void mfma_split2(float x, float y, float neg, unsigned &hi, unsigned &lo)
{
    const v2h h = __builtin_convertvector((vec2f{x, y}), v2h);
    const vec2f r = {__builtin_fmaf((float)h[0], neg, x), __builtin_fmaf((float)h[1], neg, y)};
    hi = __builtin_bit_cast(unsigned, h);
    lo = __builtin_bit_cast(unsigned, __builtin_convertvector(r, v2h));
}
typedef unsigned v4u __attribute__((ext_vector_type(4)));

// LDS bytes of a group's arrays: the B operands of its 16 pairs (nblock blocks, high and
// low halves) and the FP64 slot sums of its npos class positions, one set per wave
__host__ __device__ constexpr size_t mfma_group_lds(int nblock, int npos, int waves)
{
    return (size_t)nblock * 2 * 64 * sizeof(v8h) + (size_t)waves * npos * kMfmaPairs * sizeof(double);
}

// the slot sum of class position pos for pair jp, from the groups of matrix-core results
// (group pos / 4: D[pair][pos % 4] in lane pos % 4 + 4 (pair / 4) + 16 (pair % 4))
__device__ __forceinline__ double mfma_slot_sum(const double *sAcc, int pos, int jp)
{
    return sAcc[(pos >> 2) * 64 + (pos & 3) + 4 * (jp >> 2) + 16 * (jp & 3)];
}

// LDS bytes of k_bwd_mfma_wg with w waves: two 16-bin tiles of the element spectra
// [4 KS][16] and every wave's own arrays
__host__ __device__ constexpr size_t mfma_wg_lds(int ks, int nblock, int npos, int w)
{
    return 2 * (size_t)ks * 4 * 16 * sizeof(float2) + (size_t)w * mfma_group_lds(nblock, npos, 1);
}

// One wave's group: its pairs (lane l holds pair l % 16), their receiver and the per-pair
// coefficients F.B = f^T Amu b (earth frame through the rotations of the point, Qf, and of
// the pair, Qb); the traces are f0 + f1 + f2 and b0 + b1 + b2 (the diagonal components,
// invariant under the rotations)
template <int NDF, int NDB>
struct MfmaGroup {
    int g0, n, r, p;
    int ew;                             // the pair's weights scaled by 2^ew
    bool valid;
    float Amu[NDF][NDB];
};

// Loads group grp: its B operands into sW (the v8h at (2 block + part) 64 + l' holds part
// hi / lo of 2^ew W of pair l' % 16 and the block's component and variable, traces
// 8 (l' / 16) + q, q = 0..7; zero past the group or the 25 traces), its slot sums zeroed, its
// coefficients.  Called by the 64 lanes of each of the group's NW waves (wv: which; the
// waves share sW, each has its own sAcc); the caller synchronises before sW or sAcc is read.
template <int NDF, int NDB, int NVB, int NW>
__device__ __forceinline__ void mfma_group_setup(MfmaGroup<NDF, NDB> &G, int grp, const int *group_first,
                                                 const int *order, int R, const float *Wb, const float *Qb,
                                                 const float *Qf, const PathConf &pc, int npos, v8h *sW,
                                                 double *sAcc, int l, int wv)
{
    constexpr int J = NVB * 25;
    const int jp = l & 15, g = l >> 4;
    G.g0 = group_first[grp];
    G.n = group_first[grp + 1] - G.g0;
    // all weights loaded at once, without branches (past the traces or the group: a valid
    // weight, then zero)
    constexpr int NBLK = mfma_nblock(NDB, NVB);
    const float *wp = Wb + (size_t)(G.g0 + min(jp, G.n - 1)) * NDB * J;
    float w[NBLK][8], mx = 0.0f;
#pragma unroll
    for (int v = 0; v < NVB; ++v)
#pragma unroll
        for (int c = 0; c < NDB; ++c) {
            if (!mfma_has(NDB, v, c)) continue;
#pragma unroll
            for (int q = 0; q < 8; ++q) w[mfma_wblock(NDB, v, c)][q] = wp[c * J + 25 * v + min(8 * g + q, 24)];
        }
    // the pair's scale: its largest weight to below 2^14 (lanes jp, jp + 16, .. share it)
#pragma unroll
    for (int b = 0; b < NBLK; ++b)
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            if (jp >= G.n || 8 * g + q >= 25) w[b][q] = 0.0f;
            mx = fmaxf(mx, fabsf(w[b][q]));
        }
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    int e;
    (void)frexpf(mx, &e);
    G.ew = 14 - e;
    const float neg = mfma_neg_one();
#pragma unroll
    for (int b = 0; b < NBLK; ++b) {
        if (NW > 1 && b % NW != wv) continue;
        v4u hi, lo;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            unsigned h, o;
            mfma_split2(ldexpf(w[b][2 * q], G.ew), ldexpf(w[b][2 * q + 1], G.ew), neg, h, o);
            hi[q] = h;
            lo[q] = o;
        }
        sW[(2 * b) * 64 + l] = __builtin_bit_cast(v8h, hi);
        sW[(2 * b + 1) * 64 + l] = __builtin_bit_cast(v8h, lo);
    }
    for (int s = l; s < npos * kMfmaPairs; s += 64) sAcc[s] = 0.0;
    G.valid = jp < G.n;
    // the group's pairs share the receiver
    G.r = order[G.g0] % R;
    G.p = order[G.g0 + (G.valid ? jp : 0)] / R;                 // (no pair: the group's first point)
    if (NDF > 1) {
        float qf[6][NDF], qb[6][NDB];
#pragma unroll
        for (int i = 0; i < 6; ++i) {
#pragma unroll
            for (int m = 0; m < NDF; ++m) qf[i][m] = G.valid ? Qf[(size_t)G.p * 36 + i * 6 + m] : 0.0f;
#pragma unroll
            for (int c = 0; c < NDB; ++c) qb[i][c] = G.valid ? Qb[(size_t)(G.g0 + jp) * 36 + i * 6 + c] : 0.0f;
        }
#pragma unroll
        for (int m = 0; m < NDF; ++m)
#pragma unroll
            for (int c = 0; c < NDB; ++c) {
                float a = 0.0f;
#pragma unroll
                for (int i = 0; i < 6; ++i) a += qf[i][m] * qb[i][c];
                G.Amu[m][c] = a;
            }
    } else {
        G.Amu[0][0] = 1.0f;
    }
}

// A wave's window spectra and slot sums: per group of 4 class positions (one class), lane l
// reads column l % 4's spectrum at the bins of its pair (hoff: bytes from the receiver's
// first row to the row and the lane's bins) and holds D[pair][column] (mfma_slot_sum's
// layout).  The first NG groups' sums stay in registers across the tiles, further ones in
// LDS.  NG: that of the receiver with most groups, even, up to mfma_reg_groups; a receiver
// with fewer leaves the pairs of groups past its own out (of an odd last pair, one is summed
// into values nobody reads).  The x and y products have a sum each: two chains of dependent
// products.
constexpr int kMfmaMaxRegGroups = 8;

// Groups of a form's kernel in registers.  With 4 backward components more than these do not
// fit the 256 registers of 2 waves a SIMD and spill in every tile, which costs more than
// sums in LDS: 400 tets, 10 receivers, nt 2048, 16 + 16 slots (8 groups): 9.9 ms with 8
// groups in registers and 8.1 with 6 (4 forward components), 14.4 and 9.7 with 4 (6 forward
// components; 12 + 12 slots: 9.6 with 6 groups in registers, 8.3 with 4).  Trace-only
// kernels keep 8 (3 registers spilled with 3 variables: 12.6 ms at 8 groups against 13.3
// with 6 in registers), and 6 backward components, at one wave a SIMD, hold 8 as well.
__host__ __device__ constexpr int mfma_reg_groups(int ndf, int ndb)
{
    return ndb == 4 ? (ndf == 6 ? 4 : 6) : kMfmaMaxRegGroups;
}

template <int NG>
struct MfmaSlots {
    int ng, e0, e1;                       // groups; end of the lambda and of the mu class
    unsigned hoff[NG];
    double accx[NG], accy[NG];
};

template <int NG>
__device__ __forceinline__ void mfma_slots_init(MfmaSlots<NG> &S, const RecDesc &rd, int l, int fs)
{
    S.ng = rd.cls_end[2] >> 2;
    S.e0 = rd.cls_end[0] >> 2;
    S.e1 = rd.cls_end[1] >> 2;
#pragma unroll
    for (int g = 0; g < NG; ++g) {
        S.hoff[g] = (unsigned)((g < S.ng ? rd.cls_h[4 * g + (l & 3)] : 0) * fs + 4 * (l >> 4)) * 8u;
        S.accx[g] = S.accy[g] = 0.0;
    }
}

// loads at a byte offset from a uniform base (one scalar base, 32-bit lane offsets)
typedef const char __attribute__((address_space(1))) gchar;
__device__ __forceinline__ float2 gload2_at(const float2 *base, unsigned off)
{
    const vec2f v = *(gvec2f *)((gchar *)base + off);
    return make_float2(v.x, v.y);
}
__device__ __forceinline__ float4 gload4_at(const float2 *base, unsigned off)
{
    const vec4f v = *(gvec4f *)((gchar *)base + off);
    return make_float4(v.x, v.y, v.z, v.w);
}

// dx + dy + sum over the tile's 16 bins of Re(bk H) = bk.x H.x + bk.y (-H.y) for a group's 4
// columns: fp32 base kernels and window spectra multiply exactly in FP64 and the products
// are summed in FP64, v_mfma_f64_4x4x4_4b_f64 (4 blocks of 4 pairs, K the 4 bins of lanes
// l / 16).  A operands: bk of pair l % 16 at bins kb .. kb + 3; B: column l % 4's spectrum
// there.
__device__ __forceinline__ void mfma_slot_group(const double (&ax)[4], const double (&ay)[4], float4 q0, float4 q1,
                                                double &dx, double &dy)
{
    const double hx[4] = {q0.x, q0.z, q1.x, q1.z}, hy[4] = {q0.y, q0.w, q1.y, q1.w};
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        dx = __builtin_amdgcn_mfma_f64_4x4x4f64(ax[v], hx[v], dx, 0, 0, 0);
        dy = __builtin_amdgcn_mfma_f64_4x4x4f64(ay[v], hy[v], dy, 0, 0, 0);
    }
}

// the base kernels of class cls (0 lambda, 1 mu, 2 mu - 2 lambda; uniform) in FP64.  (The
// empty asm keeps the branches: selects between all three classes cost more than a class.)
__device__ __forceinline__ void mfma_class(const float2 (&bk0)[4], const float2 (&bk1)[4], int cls, double (&ax)[4],
                                           double (&ay)[4])
{
    if (cls == 0) {
        asm volatile("");
#pragma unroll
        for (int v = 0; v < 4; ++v) { ax[v] = bk0[v].x; ay[v] = bk0[v].y; }
    } else if (cls == 1) {
        asm volatile("");
#pragma unroll
        for (int v = 0; v < 4; ++v) { ax[v] = bk1[v].x; ay[v] = bk1[v].y; }
    } else {
        asm volatile("");
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            ax[v] = __builtin_fma((double)bk0[v].x, -2.0, (double)bk1[v].x);
            ay[v] = __builtin_fma((double)bk0[v].y, -2.0, (double)bk1[v].y);
        }
    }
}

// this lane's forward spectra of tile t (pair l % 16's point, bins 16 t + 4 (l / 16) .. + 3).
// A lane without a pair loads the group's first point (no branch): its weights are zero, so
// its base kernels and rows of the slot sums are zero, and nothing reads them.
template <int NDF>
__device__ __forceinline__ void mfma_load_f(const float2 *Fp, int l, int t, float4 (&f4)[NDF][2])
{
    const float4 *src = reinterpret_cast<const float4 *>(Fp + (size_t)t * (16 * NDF) + 4 * (l >> 4));
#pragma unroll
    for (int m = 0; m < NDF; ++m) {
        f4[m][0] = src[8 * m];
        f4[m][1] = src[8 * m + 1];
    }
}

// this lane's element spectra of tile t: variable v's trace 8 (l / 16) + q in a[8 v + q], bin
// 16 t + l % 16 (past the 25 traces: the last one, whose B operands there are zero).  uoff:
// bytes to the traces of variable 0 (mfma_uoff)
__device__ __forceinline__ void mfma_uoff(int l, unsigned (&uoff)[8])
{
#pragma unroll
    for (int q = 0; q < 8; ++q) uoff[q] = (unsigned)(min(8 * (l >> 4) + q, 24) * 16 + (l & 15)) * 8u;
}
template <int NVB>
__device__ __forceinline__ void mfma_load_u(const float2 *Ue, const unsigned (&uoff)[8], int t, float2 (&a)[8 * NVB])
{
    const float2 *Ut = Ue + (size_t)t * (16 * 25 * NVB);
#pragma unroll
    for (int v = 0; v < NVB; ++v)
#pragma unroll
        for (int q = 0; q < 8; ++q) a[8 * v + q] = gload2_at(Ut, uoff[q] + 25u * 16u * 8u * v);
}

// One 16-bin tile t of a group, given its element spectra a: the matrix cores give every
// pair's NDB carried backward components at the tile's 16 bins (real and imaginary parts
// as two products); lane l then holds pair l % 16 at bins kb = 16 t + 4 (l / 16) .. + 3 and
// forms the base kernels with the forward spectra f4 of the pair's point; then the slot
// sums Re(bk H) with the receiver's window spectra on the FP64 matrix cores.  next_u and
// next_f load the next tile's spectra into a and f4 once they are used.  MORE: receivers may
// have more than NG groups of slots.
template <int NDF, int NDB, int NVB, int NG, bool MORE, class NextU, class NextF>
__device__ __forceinline__ void mfma_tile(const MfmaGroup<NDF, NDB> &G, MfmaSlots<NG> &S, float2 (&a)[8 * NVB],
                                          float4 (&f4)[NDF][2], const v8h *sW, double *sAcc, int l, int t,
                                          const PathConf &pc, const RecDesc &rd, const float2 *Hr, NextU &&next_u,
                                          NextF &&next_f)
{
    constexpr int KS = 8 * NVB, PF = NG < 4 ? NG : 4;          // window spectra of PF groups loaded ahead
    // Loads complete in the order they are issued, so they are issued in the order of their
    // use: this tile's window spectra, then the next tile's element spectra (when this
    // tile's are split) and forward spectra (when this tile's are multiplied).
    const float2 *Ht = Hr + (t << 4);
    float4 h[PF][2];
#pragma unroll
    for (int g = 0; g < PF; ++g) {
        h[g][0] = gload4_at(Ht, S.hoff[g]);
        h[g][1] = gload4_at(Ht, S.hoff[g] + 16u);
    }
    __builtin_amdgcn_sched_barrier(0);
    v4f accR[NDB], accI[NDB];
#pragma unroll
    for (int c = 0; c < NDB; ++c) {
        accR[c] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
        accI[c] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
    }
    // the tile's scale: its largest |U| to below 2^14
    float mx = 0.0f;
#pragma unroll
    for (int s = 0; s < KS; ++s) mx = mfma_max3(mx, a[s].x, a[s].y);
    mx = mfma_wave_max(mx);
    int e;
    (void)frexpf(mx, &e);
    int eu = __builtin_amdgcn_readfirstlane(14 - e);
    if (eu > 126) {                                            // (beyond a float's power of two)
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            a[s].x = ldexpf(a[s].x, eu - 126);
            a[s].y = ldexpf(a[s].y, eu - 126);
        }
    }
    const float us = ldexpf(1.0f, min(eu, 126)), neg = mfma_neg_one();
#pragma unroll
    for (int v = 0; v < NVB; ++v) {
        v4u h4[4];                                             // re hi, re lo, im hi, im lo
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            unsigned h, o;
            mfma_split2(a[8 * v + 2 * q].x * us, a[8 * v + 2 * q + 1].x * us, neg, h, o);
            h4[0][q] = h;
            h4[1][q] = o;
            mfma_split2(a[8 * v + 2 * q].y * us, a[8 * v + 2 * q + 1].y * us, neg, h, o);
            h4[2][q] = h;
            h4[3][q] = o;
        }
        const v8h rh = __builtin_bit_cast(v8h, h4[0]), rl = __builtin_bit_cast(v8h, h4[1]);
        const v8h ih = __builtin_bit_cast(v8h, h4[2]), il = __builtin_bit_cast(v8h, h4[3]);
#pragma unroll
        for (int c = 0; c < NDB; ++c) {
            if (!mfma_has(NDB, v, c)) continue;
            const int b = mfma_wblock(NDB, v, c);
            const v8h wh = sW[(2 * b) * 64 + l], wl = sW[(2 * b + 1) * 64 + l];
            accR[c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(rh, wh, accR[c], 0, 0, 0);
            accI[c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ih, wh, accI[c], 0, 0, 0);
            accR[c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(rh, wl, accR[c], 0, 0, 0);
            accI[c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ih, wl, accI[c], 0, 0, 0);
            accR[c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(rl, wh, accR[c], 0, 0, 0);
            accI[c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(il, wh, accI[c], 0, 0, 0);
        }
    }
    next_u(a);
    __builtin_amdgcn_sched_barrier(0);
    // base kernels of this lane's pair at bins kb + v, scaled back (column l % 16: this
    // lane's pair)
    const int es = -(eu + G.ew);
    float2 bk0[4], bk1[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
#pragma clang fp contract(fast)
        float2 f[NDF], b[NDB];
#pragma unroll
        for (int m = 0; m < NDF; ++m)
            f[m] = (v & 1) ? make_float2(f4[m][v >> 1].z, f4[m][v >> 1].w) : make_float2(f4[m][v >> 1].x, f4[m][v >> 1].y);
#pragma unroll
        for (int c = 0; c < NDB; ++c) b[c] = make_float2(accR[c][v], accI[c][v]);
        if constexpr (NDF == 1) {
            const float2 pr = cmulf(f[0], b[0]);
            bk0[v] = make_float2(ldexpf(-pr.x, es), ldexpf(-pr.y, es));
            bk1[v] = make_float2(ldexpf(-pr.x, es + 1), ldexpf(-pr.y, es + 1));
        } else {
            const float2 trf = make_float2(f[0].x + f[1].x + f[2].x, f[0].y + f[1].y + f[2].y);
            const float2 trb = make_float2(b[0].x + b[1].x + b[2].x, b[0].y + b[1].y + b[2].y);
            const float2 lam = cmulf(trf, trb);
            bk0[v] = make_float2(ldexpf(-lam.x, es), ldexpf(-lam.y, es));
            // (mu: full strain is carried only when some kernel reads it)
            float2 mu = make_float2(0.f, 0.f);
#pragma unroll
            for (int m = 0; m < NDF; ++m) {
                float2 gm = make_float2(G.Amu[m][0] * b[0].x, G.Amu[m][0] * b[0].y);
#pragma unroll
                for (int c = 1; c < NDB; ++c) { gm.x += G.Amu[m][c] * b[c].x; gm.y += G.Amu[m][c] * b[c].y; }
                mu.x += f[m].x * gm.x;
                mu.x -= f[m].y * gm.y;
                mu.y += f[m].x * gm.y;
                mu.y += f[m].y * gm.x;
            }
            bk1[v] = make_float2(ldexpf(-mu.x, es + 1), ldexpf(-mu.y, es + 1));
        }
    }
    // (the base kernels before the loads: loads moved above the last use of their registers'
    // present values go to other registers, waited for and copied at the end of the tile)
    asm volatile("" ::"v"(bk0[0].x), "v"(bk0[0].y), "v"(bk0[1].x), "v"(bk0[1].y), "v"(bk0[2].x), "v"(bk0[2].y),
                 "v"(bk0[3].x), "v"(bk0[3].y), "v"(bk1[0].x), "v"(bk1[0].y), "v"(bk1[1].x), "v"(bk1[1].y),
                 "v"(bk1[2].x), "v"(bk1[2].y), "v"(bk1[3].x), "v"(bk1[3].y) : "memory");
    next_f(f4);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    // slot sums, group by group; the base kernels are converted once per class
    double ax[4], ay[4];
    mfma_class(bk0, bk1, S.e0 > 0 ? 0 : (S.e1 > 0 ? 1 : 2), ax, ay);
#pragma unroll
    for (int g = 0; g < NG; ++g) {
        if (g > 0 && (g & 1) == 0 && g >= S.ng) break;
        if (g > 0 && (g == S.e0 || g == S.e1)) mfma_class(bk0, bk1, g < S.e1 ? 1 : 2, ax, ay);
        const float4 q0 = h[g % PF][0], q1 = h[g % PF][1];
        if (g + PF < NG) {
            const unsigned off = S.hoff[g + PF < NG ? g + PF : 0];
            h[g % PF][0] = gload4_at(Ht, off);
            h[g % PF][1] = gload4_at(Ht, off + 16u);
        }
        mfma_slot_group(ax, ay, q0, q1, S.accx[g], S.accy[g]);
    }
    if constexpr (MORE)
        for (int g = NG; g < S.ng; ++g) {
            const unsigned off = (unsigned)(rd.cls_h[4 * g + (l & 3)] * pc.fstride + 4 * (l >> 4)) * 8u;
            const float4 q0 = gload4_at(Ht, off), q1 = gload4_at(Ht, off + 16u);
            mfma_class(bk0, bk1, g < S.e0 ? 0 : (g < S.e1 ? 1 : 2), ax, ay);
            double dx = sAcc[g * 64 + l], dy = 0.0;
            mfma_slot_group(ax, ay, q0, q1, dx, dy);
            sAcc[g * 64 + l] = dx + dy;
        }
}

// the register groups into sAcc (before the lanes read each other's sums)
template <int NG>
__device__ __forceinline__ void mfma_store_slots(const MfmaSlots<NG> &S, int l, double *sAcc)
{
#pragma unroll
    for (int g = 0; g < NG; ++g)
        if (g < S.ng) sAcc[g * 64 + l] = S.accx[g] + S.accy[g];
}

// Physical kernels (kernel.f90:665-832) of the group's pairs with the model at the point,
// after the damping of every receiver processed in this step (readfields.f90:3184-3204).
// Called by all lanes of the group's NW waves: lane l serves pair l % 16 and every 4 NW-th
// kernel from 4 wv + l / 16 on.  phys: [point][nk]; base_out (optional): [point][nk][6]
template <int NDF, int NDB, int NW>
__device__ __forceinline__ void mfma_finish(const MfmaGroup<NDF, NDB> &G, int l, int wv, const double *sAcc,
                                            const PathConf &pc, const RecDesc &rd, const KernDesc *kern,
                                            const int *model_idx, const float *model, int ndepth, int relative,
                                            int nk, double *phys, double *base_out, const double *xyz,
                                            const uint8_t *active, int P, int R, const double *rec_xyz)
{
    if (!G.valid) return;
    const int p = G.p, r = G.r, jp = l & 15;
    const int mi = model_idx[p];
    const float vp = model[0 * ndepth + mi], vs = model[1 * ndepth + mi], rho_f = model[2 * ndepth + mi];
    const double rho = rho_f;
    double damp = 1.0;
    if (pc.damp_radius > 0.0 && active) {
        const double x0 = xyz[3 * (size_t)p], x1 = xyz[3 * (size_t)p + 1], x2 = xyz[3 * (size_t)p + 2];
        const double ds = sqrt((x0 - pc.src_r[0]) * (x0 - pc.src_r[0]) + (x1 - pc.src_r[1]) * (x1 - pc.src_r[1])
                               + (x2 - pc.src_r[2]) * (x2 - pc.src_r[2]));
        const double fsrc = ds < pc.damp_radius ? ds / pc.damp_radius : 1.0;
        for (int r2 = r; r2 < R; ++r2) {
            if (!active[(size_t)(p / P) * R + r2]) continue;
            const double *c = rec_xyz + 3 * r2;
            const double dr = sqrt((x0 - c[0]) * (x0 - c[0]) + (x1 - c[1]) * (x1 - c[1]) + (x2 - c[2]) * (x2 - c[2]));
            damp = damp * (dr < pc.damp_radius ? dr / pc.damp_radius : 1.0) * fsrc;
        }
    }
    for (int kk = 4 * wv + (l >> 4); kk < rd.nkernel; kk += 4 * NW) {
        const int k = rd.first_kernel + kk;
        const KernDesc &kd = kern[k];
        double b[kNumBk];
#pragma unroll
        for (int qq = 0; qq < kNumBk; ++qq)
            b[qq] = kd.slot[qq] >= 0 ? mfma_slot_sum(sAcc, rd.cls_pos[kd.slot[qq]], jp) * damp : 0.0;
        if (base_out) {
            for (int qq = 0; qq < 6; ++qq) base_out[((size_t)p * nk + k) * 6 + qq] = b[qq];
            continue;
        }
        double v = 0.0;
        switch (kd.param) {
        case 0: v = relative ? b[0] * (double)(rho_f * (vp * vp - 2 * (vs * vs))) : b[0]; break;
        case 3: v = relative ? b[1] * (double)(rho_f * (vs * vs)) : b[1]; break;
        case 1: v = relative ? 2.0 * rho * (double)(vp * vp) * b[0] : 2.0 * rho * (double)vp * b[0]; break;
        case 2: v = (relative ? 2.0 * rho * (double)(vs * vs) : 2.0 * rho * (double)vs) * b[6]; break;
        default: v = 0.0;
        }
        phys[(size_t)p * nk + k] = v;
    }
}

// ------------------------------------------------------------------------------------
// k_bwd_mfma: one workgroup of 4 waves per group of at most 16 pairs of one (element,
// receiver), groups of element runs u0 .. u0 + ubatch - 1 (the others are left to another
// launch).  The waves share the group's weights and take its 16-bin tiles in turn; their
// slot sums are added at the end.  Only the lambda and mu base kernels (and mu - 2 lambda)
// are formed: the host sends kernel sets with anisotropic parameters to k_bwd_eval.  Hp:
// window spectra, rows fstride apart, zero past nomega; F: forward spectra (tile_at), zero
// past nomega.  xcd: groups in XCD-contiguous ranges (the groups of an element on one XCD).
// Bound: by the forward and element spectra, 4 NDF 128-byte lines a pair and 8-bin row (76
// GB read a launch of 20 ms, 3.8 TB/s, over 50,000 tets x 10 receivers), and by the latency
// of the wave's instructions in between (vector units 39 % and matrix units 17 % busy there:
// splitting, base kernels and slot sums) at the 2 waves a SIMD that 201 to 256 registers
// leave (1 with 6 backward components); 3 waves spill and were slower (12.8 against 9.8 ms a
// launch).  Tiles contiguous in memory, zero (component, variable) blocks left out, and the
// slot sums on the FP64 matrix units (4 x 4 x 4, a group of 4 slots and 4 bins a product) in
// place of FP64 vector products: 357 -> 311 ms (12,000 tets, 10 receivers, nt 2048), 124 ->
// 88 ms (40 voxels, 200 receivers, nt 4096), 428 -> 417 ms (100 tets, 50 receivers, 24 slots a
// receiver).  Four waves a group against one: 311 against 294, 88 against 89 and 417 against
// 460 ms (one wave's 6 register groups of slots spilled): four lose 6 % where groups abound
// and gain where they are few.
// ------------------------------------------------------------------------------------
template <int NDF, int NDB, int NVB, int NG>
__global__ __launch_bounds__(64 * kMfmaWaves, NDB <= 4 ? 2 : 1) void k_bwd_mfma(
    PathConf pc, int u0, int ubatch, int ngroups, const int *group_first, const int *group_erun,
    const float2 *U, const int *order, int R, const float *Wb, const float *Qb, const float *Qf,
    const float2 *F, const RecDesc *recs, const KernDesc *kern, const float2 *Hp, int npos,
    const int *model_idx, const float *model, int ndepth, int relative, int nk, double *phys, double *base_out,
    const double *xyz, const uint8_t *active, int P, const double *rec_xyz, int xcd)
{
    constexpr int J = NVB * 25, KS = mfma_ks(NVB), NW = kMfmaWaves;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const int grp = xcd ? xcd_block_n(ngroups) : ((int)blockIdx.x < ngroups ? (int)blockIdx.x : -1);
    if (grp < 0) return;
    const int eu = group_erun[grp];
    if (eu < u0 || eu >= u0 + ubatch) return;
    const int l = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    v8h *sW = reinterpret_cast<v8h *>(smem_raw);
    double *sSum = reinterpret_cast<double *>(sW + mfma_nblock(NDB, NVB) * 2 * 64);
    double *sAcc = sSum + (size_t)wv * npos * kMfmaPairs;
    MfmaGroup<NDF, NDB> G;
    mfma_group_setup<NDF, NDB, NVB, NW>(G, grp, group_first, order, R, Wb, Qb, Qf, pc, npos, sW, sAcc, l, wv);
    __syncthreads();
    const float2 *Ue = U + (size_t)(eu - u0) * J * pc.ustride;
    const RecDesc &rd = recs[G.r];
    const float2 *Fp = F + (size_t)G.p * NDF * pc.fstride;
    const int ntile = (pc.nomega + 15) >> 4;
    MfmaSlots<NG> S;
    mfma_slots_init(S, rd, l, pc.fstride);
    const float2 *Hr = Hp + (size_t)rd.h0 * pc.fstride;
    unsigned uoff[8];
    mfma_uoff(l, uoff);
    // the next tile's element and forward spectra are loaded into the registers of this
    // tile's as soon as those are used
    float2 a[KS];
    float4 f4[NDF][2];
    mfma_load_u<NVB>(Ue, uoff, min(wv, ntile - 1), a);
    mfma_load_f<NDF>(Fp, l, min(wv, ntile - 1), f4);
    for (int t = wv; t < ntile; t += NW) {
        const int tn = t + NW < ntile ? t + NW : t;
        mfma_tile<NDF, NDB, NVB, NG, NG == mfma_reg_groups(NDF, NDB)>(G, S, a, f4, sW, sAcc, l, t, pc, rd, Hr,
                                 [&](float2 (&x)[KS]) { mfma_load_u<NVB>(Ue, uoff, tn, x); },
                                 [&](float4 (&x)[NDF][2]) { mfma_load_f<NDF>(Fp, l, tn, x); });
    }
    mfma_store_slots(S, l, sAcc);
    __syncthreads();
    // the waves' sums of every class position
    for (int i = (int)threadIdx.x; i < S.ng * 64; i += 64 * NW) {
        double d = sSum[i];
#pragma unroll
        for (int w = 1; w < NW; ++w) d += sSum[(size_t)w * npos * kMfmaPairs + i];
        sSum[i] = d;
    }
    __syncthreads();
    mfma_finish<NDF, NDB, NW>(G, l, wv, sSum, pc, rd, kern, model_idx, model, ndepth, relative, nk, phys, base_out, xyz,
                              active, P, R, rec_xyz);
}

// ------------------------------------------------------------------------------------
// k_bwd_mfma_wg: the same evaluation with one workgroup of W waves per element run
// u0 + blockIdx.x: the waves take the run's groups W at a time (wave w: group
// erun_group_first[u] + round + w) and sweep the bins together, each 16-bin tile of the
// element's spectra loaded once into LDS for the W groups, double-buffered (the next
// tile's loads are issued before this tile's products and stored after them).  Waves
// without a group in the last round load and wait with the others.
// ------------------------------------------------------------------------------------
template <int NDF, int NDB, int NVB, int W>
__global__ __launch_bounds__(64 * W) void k_bwd_mfma_wg(
    PathConf pc, int u0, int ubatch, const int *erun_group_first, const int *group_first,
    const float2 *U, const int *order, int R, const float *Wb, const float *Qb, const float *Qf,
    const float2 *F, const RecDesc *recs, const KernDesc *kern, const float2 *Hp, int npos,
    const int *model_idx, const float *model, int ndepth, int relative, int nk, double *phys, double *base_out,
    const double *xyz, const uint8_t *active, int P, const double *rec_xyz)
{
    constexpr int J = NVB * 25, KS = mfma_ks(NVB), TILE = KS * 4 * 16; // float2 per tile
    constexpr int PER = (TILE + 64 * W - 1) / (64 * W), NBLK = mfma_nblock(NDB, NVB);
    extern __shared__ __align__(16) unsigned char smem_raw[];
    if ((int)blockIdx.x >= ubatch) return;
    const int u = u0 + (int)blockIdx.x;
    const int tid = threadIdx.x, wv = tid >> 6, l = tid & 63, jp = l & 15, bq = l >> 4;
    float2 *sU = reinterpret_cast<float2 *>(smem_raw);                  // [2][32 NVB][16]
    v8h *sW = reinterpret_cast<v8h *>(sU + 2 * TILE) + (size_t)wv * NBLK * 2 * 64;
    double *sAcc = reinterpret_cast<double *>(reinterpret_cast<v8h *>(sU + 2 * TILE) + (size_t)W * NBLK * 2 * 64)
                 + (size_t)wv * npos * kMfmaPairs;
    const float2 *Ue = U + (size_t)(u - u0) * J * pc.ustride;
    const int gbeg = erun_group_first[u], gend = erun_group_first[u + 1];
    const int ntile = (pc.nomega + 15) >> 4;
    // element spectra of row idx / 16 of tile t (row: 32 v + trace), zero past the 25 traces
    auto load = [&](int idx, int t) {
        const int v = idx >> 9, n = (idx >> 4) & 31;
        return n < 25 ? Ue[((size_t)t * J + 25 * v + n) * 16 + (idx & 15)] : make_float2(0.0f, 0.0f);
    };
    for (int round = gbeg; round < gend; round += W) {
        const int grp = round + wv;
        const bool mine = grp < gend;                                  // uniform in the wave
        MfmaGroup<NDF, NDB> G;
        if (mine)
            mfma_group_setup<NDF, NDB, NVB, 1>(G, grp, group_first, order, R, Wb, Qb, Qf, pc, npos, sW, sAcc, l, 0);
        // tile 0 (the previous round's readers of both buffers are past the last barrier)
        for (int i = 0; i < PER; ++i) {
            const int idx = tid + i * 64 * W;
            if (idx < TILE) sU[idx] = load(idx, 0);
        }
        __syncthreads();
        const RecDesc &rd = recs[mine ? G.r : 0];
        const float2 *Fp = F + (size_t)(mine ? G.p : 0) * NDF * pc.fstride;
        MfmaSlots<kMfmaMaxRegGroups> S;
        mfma_slots_init(S, rd, l, pc.fstride);
        const float2 *Hr = Hp + (size_t)rd.h0 * pc.fstride;
        for (int t = 0; t < ntile; ++t) {
            float2 nx[PER];
            const bool more = t + 1 < ntile;
            if (more) {
#pragma unroll
                for (int i = 0; i < PER; ++i) {
                    const int idx = tid + i * 64 * W;
                    nx[i] = idx < TILE ? load(idx, t + 1) : make_float2(0.0f, 0.0f);
                }
            }
            if (mine) {
                const float2 *tile = sU + (t & 1) * TILE;
                float2 a[KS];
#pragma unroll
                for (int s = 0; s < KS; ++s) a[s] = tile[(32 * (s >> 3) + 8 * bq + (s & 7)) * 16 + jp];
                float4 f4[NDF][2];
                mfma_load_f<NDF>(Fp, l, t, f4);
                mfma_tile<NDF, NDB, NVB, kMfmaMaxRegGroups, true>(G, S, a, f4, sW, sAcc, l, t, pc, rd, Hr, [](float2 (&)[KS]) {},
                                         [](float4 (&)[NDF][2]) {});
            }
            if (more) {
                float2 *nt = sU + ((t + 1) & 1) * TILE;
#pragma unroll
                for (int i = 0; i < PER; ++i) {
                    const int idx = tid + i * 64 * W;
                    if (idx < TILE) nt[idx] = nx[i];
                }
            }
            __syncthreads();
        }
        if (mine) mfma_store_slots(S, l, sAcc);
        __syncthreads();                                               // the lanes' slot sums
        if (mine)
            mfma_finish<NDF, NDB, 1>(G, l, 0, sAcc, pc, rd, kern, model_idx, model, ndepth, relative, nk, phys, base_out,
                                  xyz, active, P, R, rec_xyz);
        __syncthreads();
    }
}

}  // namespace mck
