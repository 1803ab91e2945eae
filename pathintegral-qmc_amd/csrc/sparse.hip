// Parallel sweep of sparse problems with real couplings (at most
// kSparseMaxRow nonzero entries per row, fields included): the same phases,
// arithmetic, decision classes and Philox words as the general path of
// colored.hip, so the spins are the same.
//
// What bounds it.  A row sum, a division, an exponential and Philox blocks in
// double for each of a word's P/2 attempts made the general path spend
// thousands of VALU instructions a word, in wavefronts that also waited for
// their slowest lane.  Almost all attempts do not need any of it: at the
// temperatures an anneal runs at, the energy change is far from the window in
// which a draw decides.  So a word is first decided by a filter and only what
// it leaves open is computed exactly:
//   - Filter.  With u_z = 1 where bond z of the row is unsatisfied, the energy
//     change is ediff = 4 sum u_z |J_z| - 2 sum |J_z| - 4 J_perp (1 - u_t): a
//     weighted count of unsatisfied bonds against a threshold that depends on
//     the antiparallel Trotter bonds u_t.  The weights are rounded to
//     kPlanes-bit integers and added bit-sliced, all slices of the word at once
//     (an AND, a three-input XOR and a majority per bond and plane), and the
//     sum is compared with two thresholds per u_t: above the upper one every
//     draw accepts, below the lower one (ediff < -23.5 T: exp(ediff / T) < 2^-33)
//     none does.  Both are moved outwards by the rounding of the weights and of
//     the threshold itself, so a sure answer is the exact one.
//   - Open attempts (in the window or within the rounding of its ends) go one
//     by one to a queue of the wavefront, and 64 at a time get the exact field
//     in double in row order, the exponential and their Philox bits.  The draw
//     is compared from its leading bits on with an interval around a float
//     estimate of the threshold (wider than that estimate's error); only when
//     all 32 bits leave it open is the threshold itself computed, in double.
//
// Order.  Parity 1 of color c of a sweep runs beside parity 0 of color c + 1
// (the next sweep's color 0 after the last): the two write different parities
// and colors and neither reads what the other writes, since a row reads its own
// parity in other colors and the other parity only of its own spin.  A sweep
// of n colors takes n barriers instead of 2 n, and each slot holds twice the
// words, which is what a few large replicas need.
//
// Measured against the general path: 10^3 Gaussian lattice, P=64, T=1/64, 128
// replicas, 30 traced steps 10.35 -> 0.58 ms; 80 x 80 Gaussian lattice, P=20,
// T=0.01, 32 replicas, 40 steps 18.6 -> 1.93 ms, and its 32 classical chains
// over 40 temperatures 18.6 -> 0.51 ms (32 workgroups instead of one).  Bound by
// VALU issue (77 % of the cycles of the CUs in use, 450 instructions per 64
// words on the 80 x 80 lattice; 64 % and 951 on the 10^3, whose wavefronts end
// every slot with a partly filled drain).
#include <math.h>

#include <algorithm>
#include <cmath>
#include <cstring>

#include "piqmc_internal.h"
#include "sparse.h"

namespace {

using piqmc::kSparseMaxRow;
constexpr int kPlanes = piqmc::kSparsePlanes;
constexpr int kNever = (1 << kPlanes) - 1;   // above every weighted count
constexpr int kCap = 128;                    // queue entries per wavefront (at most 63 + 64 held)

template <typename WT>
struct SparseArgs {
    int N, P, W, S, M, ncolors, R, rpw, pad0;
    uint32_t key0, key1, replica_base, sweep_base;
    const float *jperp, *temps;   // [S]
    const int *color_off;         // [ncolors + 1]
    // room only: the tables at byte 96 and J_perp at 56 is what the argument loads
    // do best with (without: 10^3, P=64, 128 replicas 440 -> 446 us; 16 x 16, P=128, 512
    // 311 -> 322; 80 x 80, P=20, 32 1816 -> 1842)
    const void *pad1[2];
    piqmc::SparseTab t;
    WT *packed;                   // [R][2][N]
    double *etrace;               // [R][S] or null
};

__device__ __forceinline__ uint32_t bop_xor(uint32_t a, uint32_t b, uint32_t c)
{
    return __builtin_amdgcn_bitop3_b32(a, b, c, 0x96);
}
__device__ __forceinline__ uint32_t bop_maj(uint32_t a, uint32_t b, uint32_t c)
{
    return __builtin_amdgcn_bitop3_b32(a, b, c, 0xE8);
}
// c ? a : b, bit by bit (operands select truth-table bits 0xF0, 0xCC, 0xAA)
__device__ __forceinline__ uint32_t bop_sel(uint32_t c, uint32_t a, uint32_t b)
{
    return __builtin_amdgcn_bitop3_b32(c, a, b, 0xCA);
}
template <typename F>
__device__ __forceinline__ uint64_t halves(F f, uint64_t a, uint64_t b, uint64_t c)
{
    return (uint64_t)f((uint32_t)a, (uint32_t)b, (uint32_t)c) |
           ((uint64_t)f((uint32_t)(a >> 32), (uint32_t)(b >> 32), (uint32_t)(c >> 32)) << 32);
}
__device__ __forceinline__ uint64_t bop_xor(uint64_t a, uint64_t b, uint64_t c)
{
    return halves([](uint32_t x, uint32_t y, uint32_t z) { return bop_xor(x, y, z); }, a, b, c);
}
__device__ __forceinline__ uint64_t bop_maj(uint64_t a, uint64_t b, uint64_t c)
{
    return halves([](uint32_t x, uint32_t y, uint32_t z) { return bop_maj(x, y, z); }, a, b, c);
}
__device__ __forceinline__ uint64_t bop_sel(uint64_t c, uint64_t a, uint64_t b)
{
    return halves([](uint32_t x, uint32_t y, uint32_t z) { return bop_sel(x, y, z); }, c, a, b);
}
// bit `bit` of pk as a word of all ones or zeros
template <typename WT>
__device__ __forceinline__ WT mask_of(uint32_t pk, int bit)
{
    return (WT)(int64_t)((int32_t)(pk << (31 - bit)) >> 31);
}

__device__ __forceinline__ int low_bit(uint32_t x) { return __ffs(x) - 1; }
__device__ __forceinline__ int low_bit(uint64_t x) { return __ffsll((unsigned long long)x) - 1; }

__device__ __forceinline__ void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// One open attempt (ediff not known to be outside the window): the decision of
// piqmc_fixed_class with the uniform of bit m of word (i, tau) in replica rep.
template <typename WT>
__device__ __forceinline__ bool decide(double ed, double T, uint32_t g, uint32_t i, uint32_t rep, int tau, int m,
                                       uint32_t k0, uint32_t k1)
{
    if (ed > 0.0) return true;
    constexpr int kPer = sizeof(WT) == 4 ? 4 : 2;  // uniform bits per Philox block
    const uint32_t c3 = (uint32_t)tau << 24;
    auto bits = [&](int qd) __attribute__((always_inline)) -> uint32_t {
        uint32_t o[4];
        philox4x32_10(g, i, rep, c3 | (uint32_t)qd, k0, k1, o);
        uint32_t v = 0;
#pragma unroll
        for (int t = 0; t < kPer; ++t) {
            const uint32_t w = sizeof(WT) == 4 ? o[t] : (m < 32 ? o[2 * t] : o[2 * t + 1]);
            v = (v << 1) | ((w >> (m & 31)) & 1u);
        }
        return v;
    };
    uint32_t u = 0;
    int nb = 0;
    if (T > 0.0 && T < INFINITY && ed <= 0.0) {
        // never accepted: exp(ed / T) < e^-23 < 2^-33
        if (ed < -23.5 * T) return false;
        // threshold 2^32 exp(ed / T) - 1/2 within 2e-5 of itself + 2 (the
        // argument is below 34, so the float exponential is within 4e-6)
        const float p = __builtin_amdgcn_exp2f((float)(ed * (1.44269504088896340736 / T))) * 4294967296.0f;
        const float mg = p * 2e-5f + 2.0f;
        const float hi = p + mg, lo = p - mg;
        const bool norej = hi >= 4294967040.0f;
        const uint32_t thi = norej ? 0xFFFFFFFFu : (uint32_t)hi + 1u, tlo = lo > 0.0f ? (uint32_t)lo : 0u;
        for (int qd = 0; qd < 32 / kPer; ++qd) {
            u |= bits(qd) << (32 - kPer - nb);
            nb += kPer;
            const uint32_t rest = nb < 32 ? 0xFFFFFFFFu >> nb : 0u;  // bits not drawn yet
            if ((u | rest) < tlo) return true;
            if (!norej && u >= thi) return false;
        }
    } else {
        for (int qd = 0; qd < 32 / kPer; ++qd, nb += kPer) u |= bits(qd) << (32 - kPer - nb);
    }
    unsigned int thr = 0;
    const int cls = piqmc_fixed_class(ed, T, &thr);
    return cls == 1 || (cls == 2 && u < thr);
}

// Places of a row in the tables, and its entries in vector loads.
template <int ZK>
constexpr int places = ZK == 6 ? 8 : ZK;
template <int ZK>
__device__ __forceinline__ void load_nb(const piqmc::SparseTab &t, int q, int (&nb)[ZK])
{
    constexpr int PL = places<ZK>;
    uint32_t v[PL / 2];
    __builtin_memcpy(v, __builtin_assume_aligned(t.nb + (size_t)q * PL, 2 * PL < 16 ? 2 * PL : 16), 2 * PL);
#pragma unroll
    for (int z = 0; z < ZK; ++z) nb[z] = (int)((v[z / 2] >> (16 * (z & 1))) & 0xffffu);
}
template <int ZK>
__device__ __forceinline__ void load_J(const piqmc::SparseTab &t, int q, float (&J)[ZK])
{
    constexpr int PL = places<ZK>;
    float v[PL];
    __builtin_memcpy(v, __builtin_assume_aligned(t.J + (size_t)q * PL, 16), 4 * PL);
#pragma unroll
    for (int z = 0; z < ZK; ++z) J[z] = v[z];
}

// Exact local field of bit m at color position q (row order, as the general
// path sums it), from the plane `mine` (whose word N is zero: fields).
template <int ZK, typename WT>
__device__ __forceinline__ double exact_field(const piqmc::SparseTab &t, int q, const WT *mine, int m)
{
    int nb[ZK];
    float J[ZK];
    load_nb<ZK>(t, q, nb);
    load_J<ZK>(t, q, J);
    double h = 0.0;
#pragma unroll
    for (int z = 0; z < ZK; ++z) {
        // J * (+-1): the sign bit flipped (padding entries add zero)
        const uint32_t sg = (uint32_t)(mine[nb[z]] >> m) << 31;
        h += (double)__uint_as_float(__float_as_uint(J[z]) ^ sg);
    }
    return h;
}

// Block-wide sum in thread 0.
__device__ __forceinline__ double block_total(double v, double *red)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    double t = 0.0;
    if (threadIdx.x == 0)
        for (int w = 0; w < (int)(blockDim.x >> 6); ++w) t += red[w];
    return t;
}

__device__ __forceinline__ int pc(uint32_t x) { return __popc(x); }
__device__ __forceinline__ int pc(uint64_t x) { return __popcll(x); }

// LDS: planes [rpw][2][N + 1] words (word N of a plane stays zero), 16 doubles,
// a queue of kCap entries per wavefront.
__host__ __device__ inline size_t sparse_planes_bytes(int N, int rpw, int wb)
{
    return ((size_t)wb * 2 * (N + 1) * rpw + 15) & ~(size_t)15;
}

template <typename WT, int ZK>
__global__ void __launch_bounds__(1024) sparse_kernel(SparseArgs<WT> a)
{
    extern __shared__ __align__(16) unsigned char smem[];
    const int N = a.N, W = a.W, tid = threadIdx.x, bd = blockDim.x, lane = tid & 63, wv = tid >> 6;
    const int r0 = blockIdx.x * a.rpw, nrep = min(a.rpw, a.R - r0), PS = N + 1;
    WT *st = reinterpret_cast<WT *>(smem);
    double *red = reinterpret_cast<double *>(smem + sparse_planes_bytes(N, a.rpw, sizeof(WT)));
    uint32_t *queue = reinterpret_cast<uint32_t *>(red + 16) + wv * kCap;
    const WT valid = W == (int)(8 * sizeof(WT)) ? ~WT(0) : ((WT(1) << W) - 1);
    WT *gst = a.packed + (size_t)r0 * 2 * N;
    for (int pl = 0; pl < 2 * nrep; ++pl) {
        for (int i = tid; i < N; i += bd) st[pl * PS + i] = gst[(size_t)pl * N + i];
        if (tid == 0) st[pl * PS + N] = 0;
    }
    const int nc = max(a.ncolors, 2);  // a problem without couplings: an empty second color
    const int segs = a.etrace ? a.S : 1, G = a.etrace ? a.M : a.S * a.M;
    __syncthreads();
    for (int seg = 0; seg < segs; ++seg) {
        // slot n: color n % nc of parity 0 in sweep n / nc, and the slot
        // before it of parity 1
        int c0 = 0, s0 = 0, m0 = 0, g0 = 0;   // color; sweep g0 of the segment = sweep m0 of its step s0
        int c1 = -1, s1 = 0, m1 = 0, g1 = -1;
        const int nslot = a.S * a.M > 0 ? G * nc + 1 : 0;
        for (int n = 0; n < nslot; ++n) {
            auto first = [&](int c) { return c < a.ncolors ? a.color_off[c] : N; };
            const bool on0 = g0 < G, on1 = g1 >= 0;
            const int b0 = on0 ? first(c0) : 0, n0 = on0 ? first(c0 + 1) - b0 : 0;
            const int b1 = on1 ? first(c1) : 0, n1 = on1 ? first(c1 + 1) - b1 : 0;
            const int t0 = (n0 + 63) & ~63, tot = t0 + n1;
            const float jp0 = a.jperp[a.etrace ? seg : s0], T0 = a.temps[a.etrace ? seg : s0];
            const float jp1 = a.jperp[a.etrace ? seg : s1], T1 = a.temps[a.etrace ? seg : s1];
            const uint32_t gg0 = a.sweep_base + (uint32_t)((a.etrace ? seg * a.M : 0) + g0);
            const uint32_t gg1 = a.sweep_base + (uint32_t)((a.etrace ? seg * a.M : 0) + g1);
            int qn = 0;  // open attempts queued by this wavefront
            // the last cnt entries: q | m << 16 | tau << 22 | replica << 23
            auto drain = [&](int cnt) __attribute__((always_inline)) {
                wave_sync();
                if (lane < cnt) {
                    const uint32_t e = queue[qn - cnt + lane];
                    const int q = (int)(e & 0xffffu), m = (int)((e >> 16) & 63u), tau = (int)((e >> 22) & 1u);
                    const int rr = (int)(e >> 23);
                    WT *mine = st + (size_t)(rr * 2 + tau) * PS;
                    const WT *other = st + (size_t)(rr * 2 + 1 - tau) * PS;
                    const int i = (int)(a.t.meta[q].x & 0xffffu);
                    const double h = exact_field<ZK, WT>(a.t, q, mine, m);
                    // slices of bit m's Trotter neighbours in the other parity
                    const int m2 = tau == 0 ? (m == 0 ? W - 1 : m - 1) : (m == W - 1 ? 0 : m + 1);
                    const WT S_ = mine[i], O = other[i];
                    const double ts = (((O >> m) & 1) ? -1.0 : 1.0) + (((O >> m2) & 1) ? -1.0 : 1.0);
                    const double jp = (double)(tau ? jp1 : jp0), T = (double)(tau ? T1 : T0);
                    const double si = ((S_ >> m) & 1) ? -1.0 : 1.0;
                    const double ed = -2.0 * si * (h + jp * ts);
                    if (decide<WT>(ed, T, tau ? gg1 : gg0, (uint32_t)i, a.replica_base + (uint32_t)(r0 + rr), tau, m,
                                   a.key0, a.key1))
                        atomicXor(reinterpret_cast<uint32_t *>(mine + i) + (m >> 5), 1u << (m & 31));
                }
                qn -= cnt;
                wave_sync();
            };
            for (int x0 = wv * 64; x0 < tot; x0 += bd) {  // wavefront-uniform: 64 words of one parity
                const int tau = x0 >= t0 ? 1 : 0;
                const int x = x0 + lane - (tau ? t0 : 0);
                const bool act = x < (tau ? n1 : n0);
                const int q = (tau ? b1 : b0) + (act ? x : 0);
                const float jp = tau ? jp1 : jp0, T = tau ? T1 : T0;
                int nb[ZK];
                load_nb<ZK>(a.t, q, nb);
                const uint4 mt = a.t.meta[q];
                const int i = (int)(mt.x & 0xffffu);
                const uint32_t neg = mt.x >> 16;
                uint32_t aw[places<ZK> / 4];
                __builtin_memcpy(aw, __builtin_assume_aligned(a.t.w + (size_t)q * (places<ZK> / 4), places<ZK>),
                                 places<ZK>);
                // thresholds on the count, per u_t: accept from pa, reject
                // below pr; T <= 0 or an infinite J_perp leaves all open.  A product
                // v or w past float's range makes the sums infinite, which leaves the
                // attempt open, or inf - inf, which the clamp makes 0: open below, and
                // accepted at two antiparallel Trotter bonds, where 4 J_perp is then
                // 1e36 times what the row could hold against it.
                uint32_t pa = 0x00ffffffu, pr = 0;
                if (T > 0.0f && T < INFINITY && fabsf(jp) < INFINITY) {
                    const float c = __uint_as_float(mt.y), v = c * jp, w = 5.875f * c * T;
                    // the sums below are rounded in float
                    const float slack = 2e-6f * (c + fabsf(v) + w + 256.0f);
                    const float ba = __uint_as_float(mt.z) + slack, br = __uint_as_float(mt.w) - w - slack;
                    auto cut = [](float x) __attribute__((always_inline)) -> uint32_t {
                        return (uint32_t)__builtin_amdgcn_fmed3f(x, 0.0f, (float)kNever);
                    };
                    pa = cut(ba + v) | (cut(ba) << 8) | (cut(ba - v) << 16);
                    pr = cut(br + v) | (cut(br) << 8) | (cut(br - v) << 16);
                }
                const int tsa = tau == 0 ? 1 : W - 1, tsb = tau == 0 ? W - 1 : 1;
                for (int rr = 0; rr < nrep; ++rr) {
                    WT unc = 0;
                    // formed here: hoisted out of this loop (one trip by
                    // default) the masks of every plane would hold registers
#pragma unroll
                    for (auto &v : aw) asm volatile("" : "+v"(v));
                    asm volatile("" : "+v"(pa), "+v"(pr));
                    if (act) {
                        WT *mine = st + (size_t)(rr * 2 + tau) * PS;
                        const WT S_ = mine[i], O = st[(size_t)(rr * 2 + 1 - tau) * PS + i];
                        WT wn[ZK];
#pragma unroll
                        for (int z = 0; z < ZK; ++z) wn[z] = mine[nb[z]];
                        // (W = 1: both Trotter neighbours are the one slice)
                        const WT Rw = W == 1 ? O : ((O << tsa) | (O >> tsb));
                        WT cnt[kPlanes];
#pragma unroll
                        for (int b = 0; b < kPlanes; ++b) cnt[b] = 0;
#pragma unroll
                        for (int z = 0; z < ZK; ++z) {
                            const WT u = bop_xor(S_, wn[z], mask_of<WT>(neg, z));
                            WT cy = 0;
#pragma unroll
                            for (int b = 0; b < kPlanes; ++b) {
                                const WT ad = u & mask_of<WT>(aw[z / 4], 8 * (z % 4) + b);
                                if (z == 0) {
                                    cnt[b] = ad;
                                } else if (b == 0) {
                                    cy = cnt[0] & ad;
                                    cnt[0] ^= ad;
                                } else {
                                    const WT c2 = bop_maj(cnt[b], ad, cy);
                                    cnt[b] = bop_xor(cnt[b], ad, cy);
                                    cy = c2;
                                }
                            }
                        }
                        const WT uL = S_ ^ O, xr = O ^ Rw;  // xr: exactly one antiparallel Trotter bond
                        WT ga = ~WT(0), gr = ~WT(0);       // count >= threshold, from the low plane up
#pragma unroll
                        for (int b = 0; b < kPlanes; ++b) {
                            const WT ta = bop_sel(xr, mask_of<WT>(pa, 8 + b),
                                                  bop_sel(uL, mask_of<WT>(pa, 16 + b), mask_of<WT>(pa, b)));
                            const WT tr = bop_sel(xr, mask_of<WT>(pr, 8 + b),
                                                  bop_sel(uL, mask_of<WT>(pr, 16 + b), mask_of<WT>(pr, b)));
                            ga = bop_maj(cnt[b], ~ta, ga);
                            gr = bop_maj(cnt[b], ~tr, gr);
                        }
                        const WT acc = ga & valid;
                        unc = gr & ~ga & valid;
                        if (acc) mine[i] = S_ ^ acc;
                    }
                    while (__ballot(unc != 0)) {
                        const bool has = unc != 0;
                        const unsigned long long bal = __ballot(has);
                        if (has) {
                            const int m = low_bit(unc);
                            unc &= unc - 1;
                            const int pos = qn + (int)__builtin_amdgcn_mbcnt_hi(
                                                     (uint32_t)(bal >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)bal, 0u));
                            queue[pos] = (uint32_t)q | ((uint32_t)m << 16) | ((uint32_t)tau << 22) | ((uint32_t)rr << 23);
                        }
                        qn += (int)__popcll(bal);
                        if (qn >= 64) drain(64);
                    }
                }
            }
            if (qn > 0) drain(qn);
            __syncthreads();
            // the next slot
            c1 = c0; s1 = s0; m1 = m0; g1 = g0;
            if (++c0 == nc) {
                c0 = 0;
                ++g0;
                if (++m0 == a.M) {
                    m0 = 0;
                    s0 = min(s0 + 1, a.S - 1);
                }
            }
        }
        if (a.etrace) {
            for (int rr = 0; rr < nrep; ++rr) {
                const WT *p0 = st + (size_t)rr * 2 * PS, *p1 = p0 + PS;
                double acc = 0.0;
                for (int q = tid; q < N; q += bd) {
                    const int i = (int)(a.t.meta[q].x & 0xffffu);
                    const WT a0 = p0[i], a1 = p1[i];
                    int nb[ZK];
                    float Jr[ZK];
                    load_nb<ZK>(a.t, q, nb);
                    load_J<ZK>(a.t, q, Jr);
#pragma unroll
                    for (int z = 0; z < ZK; ++z) {
                        const int j = nb[z];
                        const double J = (double)Jr[z];
                        const double s = (double)(a.P - 2 * (pc((WT)(a0 ^ p0[j])) + pc((WT)(a1 ^ p1[j]))));
                        acc -= (j == N ? J : 0.5 * J) * s;
                    }
                }
                const double tot = block_total(acc, red);
                if (tid == 0) a.etrace[(size_t)(r0 + rr) * a.S + seg] = tot / (double)a.P;
                __syncthreads();
            }
        }
    }
    for (int pl = 0; pl < 2 * nrep; ++pl)
        for (int i = tid; i < N; i += bd) gst[(size_t)pl * N + i] = st[pl * PS + i];
}

// Classical chains (zero Trotter coupling): no slice of a word sees another,
// so a workgroup takes `nch` chains (bits) of one parity word and the chains
// of a call spread over the device instead of sharing one workgroup per 64.
// At a preanneal's temperatures most attempts need their draw, so each is
// computed exactly at once: a lane owns a spin of one chain.
template <typename WT, int ZK>
__global__ void __launch_bounds__(1024) sparse_chains_kernel(SparseArgs<WT> a, int nch, int groups)
{
    extern __shared__ __align__(16) unsigned char smem[];
    const int N = a.N, W = a.W, tid = threadIdx.x, bd = blockDim.x;
    const int grp = blockIdx.x % groups, rt = blockIdx.x / groups, tau = rt & 1, r = rt >> 1;
    const int m0 = grp * nch, nm = min(nch, W - m0);
    WT *st = reinterpret_cast<WT *>(smem);
    WT *gst = a.packed + ((size_t)r * 2 + tau) * N;
    const WT own = (nm >= (int)(8 * sizeof(WT)) ? ~WT(0) : ((WT(1) << nm) - 1)) << m0;
    for (int i = tid; i < N; i += bd) st[i] = gst[i];
    if (tid == 0) st[N] = 0;
    __syncthreads();
    const uint32_t rep = a.replica_base + (uint32_t)r;
    for (int s = 0; s < a.S; ++s) {
        const double T = (double)a.temps[s];
        for (int m = 0; m < a.M; ++m) {
            const uint32_t g = a.sweep_base + (uint32_t)(s * a.M + m);
            for (int c = 0; c < a.ncolors; ++c) {
                const int q0 = a.color_off[c], nq = a.color_off[c + 1] - q0;
                for (int x = tid; x < nq * nm; x += bd) {
                    const int b = x / nq, q = q0 + x - b * nq, bit = m0 + b;
                    const int i = (int)(a.t.meta[q].x & 0xffffu);
                    const double h = exact_field<ZK, WT>(a.t, q, st, bit);
                    const double si = ((st[i] >> bit) & 1) ? -1.0 : 1.0;
                    const double ed = -2.0 * si * h;
                    if (decide<WT>(ed, T, g, (uint32_t)i, rep, tau, bit, a.key0, a.key1))
                        atomicXor(reinterpret_cast<uint32_t *>(st + i) + (bit >> 5), 1u << (bit & 31));
                }
                __syncthreads();
            }
        }
    }
    // this workgroup's bits of the shared words; the words were +-1 spins of
    // every chain before, of which the other workgroups own the rest
    for (int i = tid; i < N; i += bd) {
        const WT diff = (st[i] ^ gst[i]) & own;
        if constexpr (sizeof(WT) == 4) {
            if (diff) atomicXor(reinterpret_cast<unsigned int *>(gst + i), (unsigned int)diff);
        } else {
            if (diff) atomicXor(reinterpret_cast<unsigned long long *>(gst + i), (unsigned long long)diff);
        }
    }
}

template <typename WT>
SparseArgs<WT> args_of(const piqmc::SparseCall &c)
{
    const piqmc_problem *pb = c.pb;
    SparseArgs<WT> a;
    a.N = pb->N; a.P = c.P; a.W = c.P / 2; a.S = c.S; a.M = c.M; a.ncolors = pb->ncolors; a.R = c.R;
    a.rpw = c.rpw;
    a.key0 = (uint32_t)c.seed; a.key1 = (uint32_t)(c.seed >> 32);
    a.replica_base = c.rbase; a.sweep_base = c.sbase;
    a.jperp = c.jperp; a.temps = c.temps; a.color_off = c.color_off;
    a.t = pb->sparse;
    a.packed = reinterpret_cast<WT *>(c.packed);
    a.etrace = c.etrace;
    return a;
}

template <typename K, typename... A>
int launch(K kern, int grid, int block, size_t lds, hipStream_t st, A... args)
{
    PIQMC_HIP(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    kern<<<grid, block, lds, st>>>(args...);
    PIQMC_HIP(hipGetLastError());
    return PIQMC_OK;
}

template <typename WT>
int run(const piqmc::SparseCall &c, hipStream_t st)
{
    const SparseArgs<WT> a = args_of<WT>(c);
    if (c.chains) {
        const size_t lds = sizeof(WT) * (size_t)(a.N + 1);
        // chains per workgroup: few enough that the call fills the device
        // twice over (the lanes of a workgroup are spins of a color class)
        const int total = 2 * a.R * a.W;
        const int nch = std::max(1, std::min(a.W, total / 512)), groups = (a.W + nch - 1) / nch;
        switch (c.pb->sparse_rows) {
        case 4: return launch(sparse_chains_kernel<WT, 4>, 2 * a.R * groups, c.block, lds, st, a, nch, groups);
        case 6: return launch(sparse_chains_kernel<WT, 6>, 2 * a.R * groups, c.block, lds, st, a, nch, groups);
        case 8: return launch(sparse_chains_kernel<WT, 8>, 2 * a.R * groups, c.block, lds, st, a, nch, groups);
        default: return launch(sparse_chains_kernel<WT, 16>, 2 * a.R * groups, c.block, lds, st, a, nch, groups);
        }
    }
    const int grid = (a.R + a.rpw - 1) / a.rpw;
    const size_t lds = piqmc::sparse_lds(a.N, a.rpw, sizeof(WT), c.block);
    switch (c.pb->sparse_rows) {
    case 4: return launch(sparse_kernel<WT, 4>, grid, c.block, lds, st, a);
    case 6: return launch(sparse_kernel<WT, 6>, grid, c.block, lds, st, a);
    case 8: return launch(sparse_kernel<WT, 8>, grid, c.block, lds, st, a);
    default: return launch(sparse_kernel<WT, 16>, grid, c.block, lds, st, a);
    }
}

}  // namespace

namespace piqmc {

size_t sparse_lds(int N, int rpw, int word_bytes, int block)
{
    return sparse_planes_bytes(N, rpw, word_bytes) + 16 * sizeof(double) + (size_t)(block / 64) * kCap * 4;
}

int sparse_launch(const SparseCall &c, hipStream_t st)
{
    return c.P / 2 <= 32 ? run<uint32_t>(c, st) : run<uint64_t>(c, st);
}

// The tables of the problem's coloring: entries with a nonzero coupling in row
// order by color position, padded with zero couplings to 4, 6, 8 or 16.
int sparse_upload(piqmc_problem &p, const std::vector<int32_t> &order)
{
    sparse_free(p);
    const int N = p.N;
    if (N > 32767) return PIQMC_OK;
    int zmax = 0;
    for (int i = 0; i < N; ++i) {
        int z = 0;
        for (int e = 0; e < p.Z; ++e) z += p.J[(size_t)i * p.Z + e] != 0.0f;
        zmax = std::max(zmax, z);
    }
    if (zmax > kSparseMaxRow) return PIQMC_OK;
    const int ZK = zmax <= 4 ? 4 : (zmax <= 6 ? 6 : (zmax <= 8 ? 8 : 16)), PL = ZK == 6 ? 8 : ZK;
    std::vector<uint16_t> nb((size_t)PL * N, (uint16_t)N);
    std::vector<float> J((size_t)PL * N, 0.0f);
    std::vector<uint32_t> w((size_t)(PL / 4) * N, 0u);
    std::vector<uint4> meta(N);
    for (int q = 0; q < N; ++q) {
        const int i = order[q];
        double S = 0.0;
        uint32_t neg = 0;
        int z = 0;
        float *Jq = &J[(size_t)q * PL];
        for (int e = 0; e < p.Z; ++e) {
            const float v = p.J[(size_t)i * p.Z + e];
            if (v == 0.0f) continue;
            const int j = p.idx[(size_t)i * p.Z + e];
            nb[(size_t)q * PL + z] = (uint16_t)(j == i ? N : j);
            Jq[z] = v;
            if (v < 0.0f) neg |= 1u << z;
            S += fabs((double)v);
            ++z;
        }
        // Weights lrint(c |J|) whose sum stays below kNever.  The count differs
        // from c times the exact weight of the unsatisfied bonds by at least
        // the sum of the weights' negative rounding errors and at most that of
        // the positive ones; of a few scales the one whose errors are smallest
        // relative to it is taken.
        double c = 0.0, lo = 0.0, hi = 0.0, best = INFINITY;
        const double cmax = S > 0.0 ? (kNever - 1 - 0.5 * ZK) / S : 0.0;
        for (int k = 0; k < 8 && cmax > 0.0 && cmax < 1e30 && S < 1e30; ++k) {
            const double ck = (double)(float)(cmax * (1.0 - k / 64.0));
            double l = 0.0, h = 0.0;
            for (int y = 0; y < z; ++y) {
                const double x = fabs((double)Jq[y]) * ck, er = rint(x) - x;
                l += std::min(er, 0.0);
                h += std::max(er, 0.0);
            }
            if ((h - l) / ck < best) best = (h - l) / ck, c = ck, lo = l, hi = h;
        }
        // A count above c (S/2 + J_perp (1 - u_t)) + hi accepts, one below c (...
        // - 5.875 T) + lo never does; one is added for the truncation of the
        // thresholds, 0.02 keeps both strict.  Without a scale all are open.
        float f[3] = {0.0f, (float)kNever, -1e30f};
        if (c > 0.0) {
            for (int y = 0; y < z; ++y)
                w[(size_t)q * (PL / 4) + y / 4] |= (uint32_t)rint(fabs((double)Jq[y]) * c) << (8 * (y % 4));
            f[0] = (float)c;
            f[1] = (float)(0.5 * c * S + hi + 1.02);
            f[2] = (float)(0.5 * c * S + lo + 0.98);
        }
        uint32_t b[3];
        memcpy(b, f, sizeof(b));
        meta[q] = make_uint4((uint32_t)i | (neg << 16), b[0], b[1], b[2]);
    }
    // one allocation and one copy: [meta | J | w | nb], 16-byte aligned parts
    const size_t bm = meta.size() * sizeof(uint4), bj = J.size() * 4, bw = (w.size() * 4 + 15) & ~(size_t)15;
    std::vector<unsigned char> img(bm + bj + bw + nb.size() * 2);
    memcpy(img.data(), meta.data(), bm);
    memcpy(img.data() + bm, J.data(), bj);
    memcpy(img.data() + bm + bj, w.data(), w.size() * 4);
    memcpy(img.data() + bm + bj + bw, nb.data(), nb.size() * 2);
    unsigned char *d = nullptr;
    hipError_t e = hipMalloc((void **)&d, img.size());
    if (e == hipSuccess) e = hipMemcpy(d, img.data(), img.size(), hipMemcpyHostToDevice);
    if (e != hipSuccess) {
        if (d) (void)hipFree(d);
        return hip_fail(e, "problem upload");
    }
    p.d_sparse = d;
    p.sparse.meta = reinterpret_cast<const uint4 *>(d);
    p.sparse.J = reinterpret_cast<const float *>(d + bm);
    p.sparse.w = reinterpret_cast<const uint32_t *>(d + bm + bj);
    p.sparse.nb = reinterpret_cast<const uint16_t *>(d + bm + bj + bw);
    p.sparse_rows = ZK;
    return PIQMC_OK;
}

void sparse_free(piqmc_problem &p)
{
    if (p.d_sparse) (void)hipFree(p.d_sparse);
    p.d_sparse = nullptr;
    p.sparse = SparseTab();
    p.sparse_rows = 0;
}

}  // namespace piqmc
