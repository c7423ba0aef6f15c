// er_linefft.h -- PME transforms of grid lengths that have no compiled plane
// or line kernel: the same two stages as k_pme_spec2d / k_pme_axis1_t with the
// lengths and their factors as kernel arguments.  A line of length
// N = R_0 R_1 (R_2) is transformed in place in LDS, one pass per factor;
// each pass is a register DFT of one radix (er_fft.h), picked by a uniform
// branch.  The reference transforms any K1 x K2 x K3 (erdst/fft_iface.F90:38-50);
// lengths with a prime factor above 7 keep the direct kernels
// (k_pme_spec2d_gen, k_pme_axis1_gen), which cost O(N) per element.
#pragma once
#include "er_kernels.h"

// The factors of a line length for the inverse transform (decimation in
// time).  The input sits in digit order, index m = k_0 + R_0 (k_1 + R_1 k_2) at
// position k_0 len_1 + k_1 len_2 + k_2 (the rev table); pass i, from the last
// factor to the first, works on blocks of length len_i, items (block b, offset
// n < sub[i]) holding the R elements b len_i + n + sub a: the twiddle of n k,
// then the DFT.  The output is in natural order.  No value leaves its own
// item, so a pass costs one barrier.
struct LinePlan {
    int N, nf;
    int R[3], sub[3], tstep[3];   // radix, items per block, twiddle step N / len
    unsigned int msub[3];         // reciprocals of sub (fast_div)
};

// x / d for x d < 2^32, m = ceil(2^32 / d) (unused for d = 1)
__device__ __forceinline__ int fast_div(int x, int d, unsigned int m)
{
    return d == 1 ? x : (int)__umulhi((unsigned int)x, m);
}

// One pass of radix R over nline lines (line l at base + l ls, element e at
// + e es); items run lines fastest, so a wave's lanes read neighbouring lines
// (ls odd along rows, 1 along columns: no bank conflicts) and mostly one
// twiddle.  With gout the results leave for global memory instead, element e
// of line l at gout[e gs + l].
template <int R>
__device__ __forceinline__ void line_pass(float2 *base, int nline, unsigned int mline, int ls, int es, int nitem,
                                          int sub, unsigned int msub, int tstep, const float2 *tw,
                                          const float2 *__restrict__ tws, float2 *__restrict__ gout, int gs)
{
    const int NT = blockDim.x;
    for (int it = threadIdx.x; it < nitem; it += NT) {
        const int j = fast_div(it, nline, mline), l = it - j * nline;
        const int b = fast_div(j, sub, msub), n = j - b * sub;
        const int e0 = b * sub * R + n;
        float2 *p = base + l * ls + e0 * es;
        const int st = sub * es;
        float2 v[R];
#pragma unroll
        for (int a = 0; a < R; ++a) v[a] = p[a * st];
        const int e = n * tstep;  // n k tstep < sub R tstep = N
#pragma unroll
        for (int k = 1; k < R; ++k) v[k] = erfft::cmul(v[k], tw[e * k]);
        erfft::fft<R, +1>(v, tws + (R >= 4 ? tws_off(R) : 0));
        if (gout) {
#pragma unroll
            for (int a = 0; a < R; ++a) gout[(size_t)(e0 + sub * a) * gs + l] = v[a];
        } else {
#pragma unroll
            for (int a = 0; a < R; ++a) p[a * st] = v[a];
        }
    }
}

// every pass over nline lines; gout (the last pass) as in line_pass
__device__ __forceinline__ void line_dft(const LinePlan &pl, float2 *base, int nline, unsigned int mline, int ls,
                                         int es, const float2 *tw, const float2 *__restrict__ tws,
                                         float2 *__restrict__ gout = nullptr, int gs = 0)
{
    for (int i = pl.nf - 1; i >= 0; --i) {
        float2 *go = i == 0 ? gout : nullptr;
#define ER_LP(r)                                                                                           \
    case r:                                                                                                \
        line_pass<r>(base, nline, mline, ls, es, nline * (pl.N / r), pl.sub[i], pl.msub[i], pl.tstep[i], tw, \
                     tws, go, gs);                                                                         \
        break;
        switch (pl.R[i]) {
            ER_LP(2) ER_LP(3) ER_LP(4) ER_LP(5) ER_LP(6) ER_LP(7) ER_LP(8) ER_LP(9) ER_LP(10) ER_LP(12) ER_LP(15)
            ER_LP(16)
        }
#undef ER_LP
        __syncthreads();
    }
}

// Forward DFT of nline mostly-zero lines (a solute's stencils), one wave per
// line, each lane summing its outputs x = lane, lane + 64, ... over the
// line's non-zero elements in order -- lds_dft_lines without the terms that
// add +-0, so its sums are the same to the last bit (the solute's self energy
// is a small difference of this transform's square sum and the real-space
// part, and keeps the digits it had).  Output x goes to position rev[x].
__device__ __forceinline__ void line_dft_sparse(float2 *base, int nline, int ls, int es, int K, unsigned int mK,
                                                const float2 *tw, const unsigned short *rev)
{
    const int lane = threadIdx.x & 63, nw = blockDim.x >> 6;
    for (int L = threadIdx.x >> 6; L < nline; L += nw) {
        float2 *line = base + L * ls;
        unsigned long long nz[4];
        bool any = false;
#pragma unroll
        for (int o = 0; o < 4; ++o) {
            const int m = lane + 64 * o;
            const float2 v = m < K ? line[m * es] : make_float2(0.f, 0.f);
            nz[o] = __ballot(v.x != 0.0f || v.y != 0.0f);
            any = any || nz[o];
        }
        if (!any) continue;  // wave-uniform
        float2 out[4];
#pragma unroll
        for (int o = 0; o < 4; ++o) {
            out[o] = make_float2(0.f, 0.f);
            if (64 * o >= K) break;
            const int x = min(lane + 64 * o, K - 1);
            float2 acc = make_float2(0.f, 0.f);
            int idx = 0, at = 0;  // idx = (at * x) mod K
            for (int q = 0; q < 4; ++q)
                for (unsigned long long t = nz[q]; t; t &= t - 1) {
                    const int m = 64 * q + __builtin_ctzll(t);
                    if (m == at + 1) {
                        idx += x;
                        if (idx >= K) idx -= K;
                    } else {
                        const int mx = __mul24(m, x);
                        idx = mx - __mul24(fast_div(mx, K, mK), K);
                    }
                    at = m;
                    const float2 v = line[m * es];
                    const float2 t2 = tw[idx];
                    const float ty = -t2.y;
                    acc.x += v.x * t2.x - v.y * ty;
                    acc.y += v.x * ty + v.y * t2.x;
                }
            out[o] = acc;
        }
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int o = 0; o < 4; ++o) {
            const int x = lane + 64 * o;
            if (x < K) line[(int)rev[x] * es] = out[o];
        }
        __builtin_amdgcn_wave_barrier();
    }
    __syncthreads();
}

// LDS bytes of k_pme_spec2d_mix: the plane (rows padded to an odd stride), both
// twiddle tables, both position tables, the self-energy partials
__host__ __device__ constexpr size_t spec2d_mix_lds(int K2, int K3)
{
    return ((size_t)K2 * (K3 | 1) + K2 + K3) * 8 + 8 * 8 + (((size_t)(K2 + K3) * 2 + 7) / 8) * 8;
}

// The product form of a plane for at most NS sites: thread (m2, g) forms the
// sites' F1(m1) F2(m2) and walks m3 = g, g + GR, ...; the NS loads of F3 are
// issued together (sites past nslt repeat the last one against a zero factor,
// which adds +-0), so a point waits for one cached line, not for one per site.
template <int NS>
__device__ __forceinline__ void plane_product(float2 *plane, int PS, const float2 *__restrict__ F, int per, int nslt,
                                              int m1, int H, int K2, int K3, unsigned int mK2,
                                              const unsigned short *r2, const unsigned short *r3,
                                              const float *__restrict__ ef, double &sp)
{
    const int tid = threadIdx.x, GR = blockDim.x / K2;  // at least one: 256 threads or more, K2 <= 256
    const int g = fast_div(tid, K2, mK2), m2 = tid - g * K2;
    if (g >= GR) return;
    float2 B[NS];
    const float2 *Fs[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        Fs[s] = F + (size_t)min(s, nslt - 1) * per;
        const float2 a = Fs[s][m1], b = Fs[s][H + m2];
        B[s] = make_float2(fmaf(a.x, b.x, -__fmul_rn(a.y, b.y)), fmaf(a.y, b.x, __fmul_rn(a.x, b.y)));
        if (s >= nslt) B[s] = make_float2(0.f, 0.f);
    }
    const int row = (int)r2[m2] * PS;
    for (int m3 = g; m3 < K3; m3 += GR) {
        const float f = ef[m3 * K2 + m2];
        float2 f3[NS], a = make_float2(0.f, 0.f);
#pragma unroll
        for (int s = 0; s < NS; ++s) f3[s] = Fs[s][H + K2 + m3];
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            // one rounding of each product pair, then the sum: the
            // association the self energy of these grids always had
            a.x = __fadd_rn(a.x, fmaf(B[s].x, f3[s].x, -__fmul_rn(B[s].y, f3[s].y)));
            a.y = __fadd_rn(a.y, fmaf(B[s].y, f3[s].x, __fmul_rn(B[s].x, f3[s].y)));
        }
        sp += self_term(f, a);
        plane[row + r3[m3]] = erfft::cscale(a, f);
    }
}

// Stage A for any K2 x K3 of small prime factors, one (insertion, m1) plane
// per workgroup: the structure factor, the FP64 half-plane self energy and the
// engfac multiply, the inverse DFT along axes 3 and 2, T[nl][m1][x2][x3].
// Few sites: the product form, stored at its place in the inverse
// transform's input order.  Many sites: each wave owns
// a block of rows, finds the sites whose stencils meet it (a ballot over 64
// sites at a time) and adds them in site order, so a point's sum has one
// order whatever the wave count; then the forward DFT over what is not zero.
// Bound by its LDS passes (a 60 x 100 plane is 48 KB: three workgroups per
// CU).  300 insertions of nine sites on 60 x 60 x 100: 412 us, the direct DFT
// 3850 us; writing T alone would take 95 us.
__global__ void __launch_bounds__(512) k_pme_spec2d_mix(int nslot, const SlotDesc *__restrict__ sd, int ord, int K1,
                                                        int K2, int K3, LinePlan p2, LinePlan p3, unsigned int mK2,
                                                        unsigned int mK3, const unsigned short *__restrict__ rev2,
                                                        const unsigned short *__restrict__ rev3, int sparse,
                                                        int n_off, const float2 *__restrict__ Ftab,
                                                        const float *__restrict__ insw,
                                                        const int4 *__restrict__ insg,
                                                        const float *__restrict__ engfac,
                                                        const float2 *__restrict__ tw2,
                                                        const float2 *__restrict__ tw3,
                                                        const float2 *__restrict__ tws, float2 *__restrict__ T,
                                                        double *__restrict__ selfpart, int ntot)
{
    extern __shared__ __align__(16) unsigned char smem[];
    const int PS = K3 | 1, NE = K2 * K3, H = K1 / 2 + 1;
    float2 *plane = reinterpret_cast<float2 *>(smem);   // [K2][PS]
    float2 *t2 = plane + (size_t)K2 * PS;                // [K2]
    float2 *t3 = t2 + K2;                                // [K3]
    double *red = reinterpret_cast<double *>(t3 + K3);   // [NT / 64]
    unsigned short *r2 = reinterpret_cast<unsigned short *>(red + 8);  // [K2]
    unsigned short *r3 = r2 + K2;                                      // [K3]
    const int m1 = blockIdx.x, nl = blockIdx.y, n = n_off + nl;
    const int tid = threadIdx.x, NT = blockDim.x, lane = tid & 63;
    float2 *Tp = T + ((size_t)nl * H + m1) * (size_t)NE;
    const int ks = ER_SLOT_OF_INS(sd, nslot, n);
    const int local = n - sd[ks].ins_off;
    if (local >= sd[ks].nins) {  // padding insertion: a zero plane and no self energy
        for (int e = tid; e < NE; e += NT) Tp[e] = make_float2(0.f, 0.f);
        if (tid == 0) selfpart[(size_t)m1 * ntot + n] = 0.0;
        return;
    }
    const int nslt = sd[ks].nslt;
    const size_t rowb = (size_t)sd[ks].site_off + (size_t)local * nslt;
    const int per = H + K2 + K3;
    for (int k = tid; k < K2; k += NT) {
        t2[k] = tw2[k];
        r2[k] = rev2[k];
    }
    for (int k = tid; k < K3; k += NT) {
        t3[k] = tw3[k];
        r3[k] = rev3[k];
    }
    const float *ef = engfac + (size_t)m1 * NE;  // [m3][m2]
    double sp = 0.0;
    if (!sparse) {
        const float2 *F = Ftab + rowb * per;
        __syncthreads();
#define ER_GEN(ns) plane_product<ns>(plane, PS, F, per, nslt, m1, H, K2, K3, mK2, r2, r3, ef, sp)
        if (nslt <= 3) ER_GEN(3);
        else if (nslt <= 6) ER_GEN(6);
        else if (nslt <= 9) ER_GEN(9);
        else ER_GEN(ER_DENSE_SITES);
#undef ER_GEN
    } else {
        for (int e = tid; e < K2 * PS; e += NT) plane[e] = make_float2(0.f, 0.f);
        __syncthreads();
        const int nw = NT >> 6, wv = tid >> 6;
        const int x0 = wv * K2 / nw, x1 = (wv + 1) * K2 / nw;  // this wave's rows
        const int np = ord * ord;
        for (int s0 = 0; s0 < nslt; s0 += 64) {
            // lane s: site s0 + s, and whether its rows g.y - c (c < ord) meet [x0, x1)
            const bool have = s0 + lane < nslt;
            const size_t my = rowb + s0 + (have ? lane : 0);
            const int4 g4 = insg[my];
            const float2 A = Ftab[my * per + m1];
            int d = g4.y - x0;
            d += (d < 0) ? K2 : 0;
            unsigned long long todo = __ballot(have && d < (x1 - x0) + ord - 1);
            while (todo) {  // wave-uniform, sites in order
                const int s = __builtin_ctzll(todo);
                todo &= todo - 1;
                const int gy = __shfl(g4.y, s, 64), gz = __shfl(g4.z, s, 64);
                const float2 a = make_float2(__shfl(A.x, s, 64), __shfl(A.y, s, 64));
                const float *w = insw + (rowb + s0 + s) * 3 * ord + ord;
                for (int p = lane; p < np; p += 64) {
                    const int c2 = p / ord, c3 = p - c2 * ord;
                    int x2 = gy - c2, x3 = gz - c3;
                    x2 += (x2 < 0) ? K2 : 0;
                    x3 += (x3 < 0) ? K3 : 0;
                    if (x2 >= x0 && x2 < x1) {
                        const float2 v = erfft::cscale(a, w[c2] * w[ord + c3]);
                        float2 *q = plane + x2 * PS + x3;
                        *q = make_float2(q->x + v.x, q->y + v.y);
                    }
                }
                // the next site's lanes may add to the same points: the wave
                // runs its LDS accesses in order, the fence keeps the compiler to it
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            }
        }
        __syncthreads();
        line_dft_sparse(plane, K2, PS, 1, K3, mK3, t3, r3);
        line_dft_sparse(plane, K3, 1, PS, K2, mK2, t2, r2);
        for (int e = tid; e < NE; e += NT) {
            const int m3 = fast_div(e, K2, mK2), m2 = e - m3 * K2;
            const float f = ef[e];
            float2 *q = plane + (int)r2[m2] * PS + r3[m3];
            const float2 a = *q;
            sp += self_term(f, a);
            *q = erfft::cscale(a, f);
        }
    }
    __syncthreads();
    line_dft(p3, plane, K2, mK2, PS, 1, t3, tws);
    line_dft(p2, plane, K3, mK3, 1, PS, t2, tws, Tp, K3);
    for (int off = 32; off > 0; off >>= 1) sp += __shfl_down(sp, off, 64);
    if (lane == 0) red[tid >> 6] = sp;
    __syncthreads();
    if (tid == 0) {
        double t = 0.0;
        for (int wv = 0; wv < (NT >> 6); ++wv) t += red[wv];
        selfpart[(size_t)m1 * ntot + n] = plane_weight(K1, m1) * t;
    }
}

// Stage B for any K1 of small prime factors, 16 interleaved insertions: the
// complex-to-real transform along axis 1 of RL = 2^rsh consecutive (x2, x3)
// lines (T and phi are both contiguous over them), RL at least 2.  Two
// neighbouring lines of one insertion share one complex transform of length
// K1: Z = X_a + i X_b over the whole Hermitian spectrum gives phi_a and phi_b as
// its real and imaginary parts, for even and odd K1 alike.  (Two insertions
// in one transform would carry a non-finite one into the other.)
// Each XCD sweeps one contiguous eighth of the blocks, so that the two halves
// of a 128-byte line of T meet in one L2.
__host__ __device__ constexpr size_t axis1_mix_lds(int K1, int RL)
{
    return ((size_t)RL * 8 * (K1 | 1) + K1) * 8 + (((size_t)K1 * 2 + 7) / 8) * 8;
}
__global__ void __launch_bounds__(256) k_pme_axis1_mix(int nchunk, int K1, int nline, int rsh, LinePlan p1,
                                                       unsigned int mL, const unsigned short *__restrict__ rev1,
                                                       const float2 *__restrict__ T, float *__restrict__ phi,
                                                       const float2 *__restrict__ tw1,
                                                       const float2 *__restrict__ tws)
{
    extern __shared__ __align__(16) unsigned char smem[];
    const int H = K1 / 2 + 1, LS = K1 | 1, RL = 1 << rsh, NP = RL >> 1, NT = blockDim.x, tid = threadIdx.x;
    const int NL = NP * 16;                             // complex lines of the block
    float2 *Z = reinterpret_cast<float2 *>(smem);       // [NP line pairs][16 insertions][LS]
    float2 *tw = Z + (size_t)NL * LS;                   // [K1]
    unsigned short *rv = reinterpret_cast<unsigned short *>(tw + K1);
    const int ngrp = (nline + RL - 1) >> rsh;
    const int total = ngrp * ((nchunk + 15) / 16), perx = (total + 7) / 8;
    const int blk = (int)(blockIdx.x & 7) * perx + (int)(blockIdx.x >> 3);
    if (blk >= total) return;
    const int tile = blk / ngrp, l0 = (blk % ngrp) << rsh;
    for (int k = tid; k < K1; k += NT) {
        tw[k] = tw1[k];
        rv[k] = rev1[k];
    }
    __syncthreads();
    // line pair q, insertion p, m: X_a, X_b -> Z(m) and Z(K1 - m)
    for (int it = tid; it < H * NL; it += NT) {
        const int q = it & (NP - 1), p = (it >> (rsh - 1)) & 15, m = it >> (rsh + 3);
        const int n = tile * 16 + p, la = l0 + 2 * q;
        const bool live = n < nchunk && la < nline;
        const float2 *src = T + ((size_t)n * H + m) * nline + la;
        const float2 a = live ? src[0] : make_float2(0.f, 0.f);
        const float2 b = live && la + 1 < nline ? src[1] : make_float2(0.f, 0.f);
        float2 *z = Z + (q * 16 + p) * LS;
        if (m == 0 || 2 * m == K1) {  // their own mirror images: real
            z[rv[m]] = make_float2(a.x, b.x);
        } else {
            z[rv[m]] = make_float2(a.x - b.y, a.y + b.x);
            z[rv[K1 - m]] = make_float2(a.x + b.y, b.x - a.y);
        }
    }
    __syncthreads();
    line_dft(p1, Z, NL, mL, LS, 1, tw, tws);
    // phi[line][x1][16]: the 16 insertions of one x1 are one 64-byte run, two per thread
    float2 *dst = reinterpret_cast<float2 *>(phi + ((size_t)tile * nline + l0) * K1 * 16);
    const int nr = min(RL, nline - l0);
    for (int q = 0; 2 * q < nr; ++q)
        for (int it = tid; it < K1 * 8; it += NT) {
            const int p = it & 7, x1 = it >> 3;
            const float2 *z = Z + (q * 16 + 2 * p) * LS + x1;
            const float2 u = z[0], v = z[LS];
            dst[(size_t)(2 * q) * K1 * 8 + it] = make_float2(u.x, v.x);
            if (2 * q + 1 < nr) dst[(size_t)(2 * q + 1) * K1 * 8 + it] = make_float2(u.y, v.y);
        }
}
