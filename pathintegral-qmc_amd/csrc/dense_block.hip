// Parallel sweep of dense couplings whose rows sum exactly in any order
// (piqmc_problem_exact_rows, symmetric rows, N <= 256), in blocks of 16 spins.
//
// What bounds it.  Every spin interacts with every other, so a slice's spins
// are decided one after the other: the time is the number of decisions in a
// row times the time of one.  With the local fields cached in LDS a decision
// still took about 1100 cycles -- an LDS read, a division and an exponential,
// two or more Philox blocks, an LDS update of the row -- and a sweep had 2 N of
// them.  Here a sweep has N, of about 410 cycles each:
//   - Draws ahead.  A uniform u does not depend on the state, so the test
//     exp(ediff / T) > u is turned into ediff > T ln(u) and the threshold is
//     ready before the decision: idle wavefronts draw the next block's Philox
//     words, transpose them (the stream stores bit b of 32 slices in a word)
//     and take the logarithm in float.  Within the float's error of the
//     threshold (a few in 10^6) the decision is made as everywhere else, in
//     double.
//   - Blocks.  One wavefront of a team decides 16 spins, a lane per slice, with
//     their fields (Trotter term included) in registers as floats: a flip
//     changes the fields of the block's later spins by one fma each.  Then all
//     wavefronts of the team apply the block's flips to the whole fields, which
//     they hold in registers in double (a lane has up to four spins of a few
//     slices; a flip adds a row of couplings, staged in LDS), and hand over the
//     next block's.  Every sum in double is exact, so the order of the additions
//     does not matter; a field within the floats' error of its threshold makes
//     the block be decided again with that spin's field summed in double.
//   - Both parities at once.  Two teams, one a parity, the odd one a block
//     behind: it reads the even parity's spins only in the block it is in, which
//     the even team has left and comes back to a whole sweep later.
// Per position of both parities, 256 spins, 4 replicas, against the cached-field
// sweep over eight wavefronts: P=16 1013 -> 169 ns, P=32 1042 -> 178 ns, P=128 1409
// -> 345 ns; 1024 replicas of P=32 4294 -> 730 ns, of P=128 9103 -> 1398 ns.  At P=32 a
// block takes 6600 cycles: 3200 to decide (16 chains of five dependent instructions,
// an LDS read of couplings each), about as long beside it for the draws, 3000 to
// apply its few flips and hand over, the rest at the two barriers.
#include <math.h>

#include <algorithm>
#include <cstring>
#include <type_traits>

#include "dense_block.h"

namespace {

using piqmc::BlockArgs;
typedef float f4 __attribute__((ext_vector_type(4)));
constexpr int kB = 16;  // spins per block: 16 decisions share two barriers and the hand-over's latency

// A team's wavefronts.  Four of each parity leave a SIMD two wavefronts and 256
// registers each, which hold a wavefront's fields (W / 4 slices of up to 256
// spins) beside the block being decided; with eight the sweep spilled, and every
// wavefront repeats the hand-over's scalar work (256 spins, P=32: 390 against
// 334 ns a position when the two were compared).
constexpr int kTeam = 4;
template <typename WT>
constexpr int kMs = 2 * (int)sizeof(WT);  // slices a wavefront holds

__device__ __forceinline__ void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The value of lane ^ J (J < 32).
template <int J>
__device__ __forceinline__ uint32_t lane_xor(uint32_t x)
{
    if constexpr (J == 1) return (uint32_t)__builtin_amdgcn_mov_dpp((int)x, 0xB1, 0xf, 0xf, true);        // quad_perm 1 0 3 2
    else if constexpr (J == 2) return (uint32_t)__builtin_amdgcn_mov_dpp((int)x, 0x4E, 0xf, 0xf, true);   // quad_perm 2 3 0 1
    else if constexpr (J == 8) return (uint32_t)__builtin_amdgcn_mov_dpp((int)x, 0x128, 0xf, 0xf, true);  // row_ror 8
    else return (uint32_t)__builtin_amdgcn_ds_swizzle((int)x, (J << 10) | 0x1f);
}

// Bit matrix across 32 lanes: lane l's bit c becomes lane c's bit l.  A step
// swaps bit J of the lane with bit J of the column: a lane keeps the half of its
// bits whose column has its own J and takes the other half from lane ^ J, moved
// by J (a rotation: what it carries round is masked).
template <int J>
__device__ __forceinline__ uint32_t transpose_step(uint32_t x, int l, uint32_t m)
{
    const uint32_t up = (uint32_t)((int32_t)(l << (31 - __builtin_ctz(J))) >> 31);  // all ones: lane has J
    const uint32_t y = lane_xor<J>(x);
    const uint32_t r = __builtin_amdgcn_alignbit(y, y, (up & (uint32_t)(2 * J - 32)) + (uint32_t)(32 - J));
    return __builtin_amdgcn_bitop3_b32(m ^ up, x, r, 0xCA);  // columns kept: x, others: r
}
__device__ __forceinline__ uint32_t transpose32(uint32_t x, int l)
{
    x = transpose_step<16>(x, l, 0x0000FFFFu);
    x = transpose_step<8>(x, l, 0x00FF00FFu);
    x = transpose_step<4>(x, l, 0x0F0F0F0Fu);
    x = transpose_step<2>(x, l, 0x33333333u);
    return transpose_step<1>(x, l, 0x55555555u);
}

template <typename WT>
__device__ __forceinline__ WT uniform(WT x)
{
    if constexpr (sizeof(WT) == 4) return (WT)__builtin_amdgcn_readfirstlane((int)x);
    else
        return (WT)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)x) |
               ((WT)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(x >> 32)) << 32);
}

template <int A, int B, typename F>
__device__ __forceinline__ void static_for(F f)
{
    if constexpr (A < B) {
        f(std::integral_constant<int, A>());
        static_for<A + 1, B>(f);
    }
}

// x with its sign bit XORed by that of s (one v_bitop3)
__device__ __forceinline__ uint32_t flip_sign(uint32_t x, uint32_t s)
{
    return __builtin_amdgcn_bitop3_b32(x, s, 0x80000000u, 0x78);
}

// LDS of a team, after the shared state words [2][blocks * kB]:
struct TeamLds {
    size_t hb, jb, rows, th, uu, fm, scratch, bytes;
};
__host__ __device__ inline TeamLds team_lds(int slots, int wb)
{
    // row pitches are the word's slices, whatever W: offsets of a block's spins
    // are then the instructions' immediates
    const size_t W = 8 * (size_t)wb;
    TeamLds t;
    size_t o = 0;
    t.hb = o;       // float [kB][W + 1] fields of the block to decide
    o += sizeof(float) * kB * (W + 1);
    t.jb = o = (o + 15) & ~(size_t)15;  // float [2][kB][kB] twice the block's couplings
    o += sizeof(float) * 2 * kB * kB;
    t.rows = o;     // float [kB][64][slots] its rows
    o += sizeof(float) * kB * 64 * slots;
    t.th = o;       // float [2][kB][W] thresholds
    o += sizeof(float) * 2 * kB * W;
    t.uu = o;       // uint32 [2][kB][W] their draws
    o += sizeof(uint32_t) * 2 * kB * W;
    t.fm = o;       // uint32 [W] a slice's flips (bit j) and old spins (bit 16 + j) in the block
    o += sizeof(uint32_t) * W;
    t.scratch = o = (o + 15) & ~(size_t)15;  // 1 KiB per wavefront: Philox words
    o += (size_t)1024 * kTeam;
    t.bytes = o;
    return t;
}
__host__ __device__ inline int N4(int N) { return (N + 3) & ~3; }
__host__ __device__ inline int blocks_of(int N) { return N > kB ? (N + kB - 1) / kB : 2; }  // two at least: see the lag
__host__ __device__ inline size_t block_lds(int N, int wb)
{
    const size_t st = ((size_t)wb * 2 * blocks_of(N) * kB + 15) & ~(size_t)15;
    return st + 16 * sizeof(double) + sizeof(int) * N4(N) + 2 * team_lds((N + 63) / 64, wb).bytes;
}

template <typename WT, int KS>
__device__ void block_sweep(const BlockArgs &a, int r, unsigned char *smem)
{
    constexpr int MS = kMs<WT>;
    const int N = a.N, W = a.W, tid = threadIdx.x, lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6), tau = wv / kTeam;
    // the deciding wavefronts (tw 0) of the two teams on different SIMDs
    const int tw = tau ? (wv + kTeam - 1) % kTeam : wv;
    const int nbk = blocks_of(N), NP = nbk * kB;
    constexpr int WP = 8 * (int)sizeof(WT), HP = WP + 1;
    WT *st = reinterpret_cast<WT *>(smem);  // [2][NP] by color position
    double *red = reinterpret_cast<double *>(smem + (((size_t)sizeof(WT) * 2 * NP + 15) & ~(size_t)15));
    const TeamLds tl = team_lds(KS, sizeof(WT));
    int *ord = reinterpret_cast<int *>(red + 16);  // [N] spins by color position
    unsigned char *base = reinterpret_cast<unsigned char *>(ord + N4(N)) + tau * tl.bytes;
    float *hb = reinterpret_cast<float *>(base + tl.hb);
    float *jb = reinterpret_cast<float *>(base + tl.jb);
    float *rows = reinterpret_cast<float *>(base + tl.rows), *th = reinterpret_cast<float *>(base + tl.th);
    uint32_t *uu = reinterpret_cast<uint32_t *>(base + tl.uu);
    uint32_t *fm = reinterpret_cast<uint32_t *>(base + tl.fm);
    uint32_t *sc = reinterpret_cast<uint32_t *>(base + tl.scratch) + 256 * tw;
    WT *mine = st + tau * NP;
    const WT *other = st + (1 - tau) * NP;
    WT *gst = reinterpret_cast<WT *>(a.packed) + (size_t)r * 2 * N;
    const uint32_t rep = a.replica_base + (uint32_t)r;

    for (int x = tid; x < 2 * NP; x += blockDim.x) {
        const int q = x % NP;
        st[x] = q < N ? gst[(size_t)(x / NP) * N + a.order[q]] : WT(0);
        if (x < N) ord[x] = a.order[x];
    }
    __syncthreads();

    // this wavefront's slices [s0, s0 + ns) of its parity and their fields:
    // f[s][k] is slice s0 + s, color position 64 k + lane
    const int per = (W + kTeam - 1) / kTeam, s0 = tw * per, ns = max(0, min(per, W - s0));
    double f[MS][KS];
#pragma unroll
    for (int s = 0; s < MS; ++s)
#pragma unroll
        for (int k = 0; k < KS; ++k) f[s][k] = 0.0;
    for (int q0 = 0; q0 < N; q0 += 4) {
        float j2[4][KS];
#pragma unroll
        for (int y = 0; y < 4; ++y)
#pragma unroll
            for (int k = 0; k < KS; ++k)
                j2[y][k] = q0 + y < N ? a.j2[((size_t)(q0 + y) * 64 + lane) * KS + k] : 0.0f;
#pragma unroll
        for (int y = 0; y < 4; ++y) {
            const uint32_t w = (uint32_t)(uniform(mine[min(q0 + y, N - 1)]) >> (ns > 0 ? s0 : 0));
#pragma unroll
            for (int s = 0; s < MS; ++s)
#pragma unroll
                for (int k = 0; k < KS; ++k)
                    f[s][k] += (double)__uint_as_float(__float_as_uint(j2[y][k]) ^ (((w >> s) & 1u) << 31));
        }
    }
#pragma unroll
    for (int k = 0; k < KS; ++k) {
        const double dg = a.diag[64 * k + lane];
#pragma unroll
        for (int s = 0; s < MS; ++s) f[s][k] = 0.5 * f[s][k] + dg;
    }

    auto finite = [](float T, float jp) { return T > 0.0f && T < INFINITY && fabsf(jp) < INFINITY; };
    // h_i + J_perp ts of block c's positions, a lane each, for the deciding
    // wavefront: this team's field before the block, the other parity's spins
    auto hand_over = [&](int c, float jp) __attribute__((always_inline)) {
        const int k0 = c * kB >> 6, l0 = (c * kB) & 63, j = lane - l0;
        if (j >= 0 && j < kB) {
            const WT O = other[c * kB + j];
            const WT Rw = tau == 0 ? (O << 1) | (O >> (W - 1)) : (W == 1 ? O : (O >> 1) | (O << (W - 1)));
            const int sh = ns > 0 ? s0 : 0;
            const uint32_t o = (uint32_t)(O >> sh), x = o ^ (uint32_t)(Rw >> sh);  // x: antiparallel neighbours
            float *hj = hb + j * HP + s0;
#pragma unroll
            for (int k = 0; k < KS; ++k) {
                if (k != k0) continue;
#pragma unroll
                for (int s = 0; s < MS; ++s)
                    if (s < ns) {
                        // J_perp ts: 0 or +-2 J_perp
                        const uint32_t b = flip_sign(__float_as_uint(2.0f * jp), o << (31 - s));
                        hj[s] = (float)f[s][k] + __uint_as_float((x >> s) & 1u ? 0u : b);
                    }
            }
        }
    };
    // twice the couplings within block c, [j][j2], a 16-byte group per lane
    auto stage_jb = [&](int c, int buf) __attribute__((always_inline)) {
        if (c * kB < N)
            reinterpret_cast<f4 *>(jb + buf * kB * kB)[lane] =
                reinterpret_cast<const f4 *>(a.jb2 + (size_t)c * kB * kB)[lane];
    };
    // the draws of 8 (32-bit words) or 4 positions of block c in sweep g, and
    // their thresholds -T ln(u) / 2 on s_i (h_i + J_perp ts)
    constexpr int kPos = sizeof(WT) == 4 ? 8 : 4, kTasks = kB / kPos;
    auto draw = [&](int task, int c, uint32_t g, float T, bool fin, int buf) __attribute__((always_inline)) {
        constexpr int kQd = 64 / kPos;  // Philox blocks per word
        const int p = lane / kQd, qd = lane % kQd, q = c * kB + task * kPos + p;
        uint32_t o[4];
        philox4x32_10(g, (uint32_t)ord[min(q, N - 1)], rep, ((uint32_t)tau << 24) | (uint32_t)qd, a.key0, a.key1, o);
        if constexpr (sizeof(WT) == 4) {
            *reinterpret_cast<uint4 *>(sc + 4 * lane) = make_uint4(o[0], o[1], o[2], o[3]);
        } else {  // halves apart: word 2 qd + t has its low slices in o[2t], its high ones in o[2t + 1]
            *reinterpret_cast<uint2 *>(sc + p * 64 + 2 * qd) = make_uint2(o[0], o[2]);
            *reinterpret_cast<uint2 *>(sc + p * 64 + 32 + 2 * qd) = make_uint2(o[1], o[3]);
        }
        wave_sync();
        const int l = lane & 31;
        constexpr int kPasses = sizeof(WT) == 4 ? 4 : 2;  // (64-bit words: the fields leave few registers)
        const float cT = fin ? -0.34657359027997264f * T : __uint_as_float(0x7fc00000u);  // NaN: decided in double
#pragma unroll kPasses
        for (int v = 0; v < 4; ++v) {
            const uint32_t u = __brev(transpose32(sc[v * 64 + lane], l));
            const int pos = sizeof(WT) == 4 ? 2 * v + (lane >> 5) : v, m = sizeof(WT) == 4 ? l : lane;
            const int x = (buf * kB + task * kPos + pos) * WP + m;  // (m >= W: places no slice reads)
            uu[x] = u;
            th[x] = cT * __builtin_amdgcn_logf(((float)u + 0.5f) * 2.3283064365386963e-10f);
        }
        wave_sync();
    };

    // The team's place: block c of sweep (step s, m of it), the index of which
    // in the call is x; `buf` holds its thresholds and block couplings.
    const int total = a.S * a.M * nbk;
    constexpr int kV = 64 * KS / 4;  // 16-byte groups per row
    int x = 0, c = 0, m = 0, s = 0, buf = 0;
    float T = total > 0 ? a.temps[0] : 0.0f, jp = total > 0 ? a.jperp[0] : 0.0f;
    if (total > 0) {
        if (tau == 0) hand_over(0, a.jperp[0]);  // the odd team's after the even one's first block
        if (tw == 1) stage_jb(0, 0);
        for (int task = tw; task < kTasks; task += kTeam)
            draw(task, 0, a.sweep_base, a.temps[0], finite(a.temps[0], a.jperp[0]), 0);
    }
    __syncthreads();
    const int segs = a.etrace ? a.S : 1, seglen = (a.etrace ? a.M : a.S * a.M) * nbk;
    for (int seg = 0; seg < segs; ++seg) {
        for (int t = 0; total > 0 && t <= seglen; ++t) {
            const bool on = tau == 0 ? t < seglen : t > 0;
            // the next place
            int cn = c + 1, mn = m, sn = s;
            if (cn == nbk) {
                cn = 0;
                if (++mn == a.M) mn = 0, ++sn;
            }
            const bool more = x + 1 < total;
            float Tn = T, jpn = jp;
            if (more && sn != s) Tn = a.temps[sn], jpn = a.jperp[sn];
            const int nq = min(kB, N - c * kB);
            if (on && tw == 0) {
                // decide the block: a lane per slice
                __builtin_amdgcn_s_setprio(3);
                // (opaque: what follows from the lane would be kept in registers
                // over the whole schedule)
                int ln = lane;
                asm volatile("" : "+v"(ln));
                const bool act = ln < W;
                const int lb = act ? ln : 0;
                // open below this distance from the threshold: the logarithm's
                // error (2e-5 of up to 11.5 T, a wide margin) and the roundings of the
                // field and of the 16 sums after it.  The field is at most bound; a sum
                // that ends near its threshold has J_perp ts within bound + 11.5 T, so
                // none exceeds 2 bound + 11.5 T: 33 half units of the last place of
                // bound, 1.97e-6, and 1.2e-5 T, which the logarithm's margin holds
                const float gd = 2.5e-4f * T + 2e-6f * a.bound;
                const float *tb = th + buf * kB * WP;
                const f4 *J = reinterpret_cast<const f4 *>(jb + buf * kB * kB);
                // the block's words, half a wavefront the low and the high slices,
                // and their transpose: bit j of a lane = spin j of its slice
                uint32_t *half = reinterpret_cast<uint32_t *>(mine + c * kB) +
                                 (sizeof(WT) == 4 ? (ln & 31) : 2 * (ln & 31) + (ln >> 5));
                const bool holds = (ln & 31) < nq && (sizeof(WT) == 8 || ln < 32);
                const uint32_t old = holds ? *half : 0u;
                const uint32_t sb = transpose32(old, ln & 31);
                uint32_t ab = 0;        // flips
                float dmin = INFINITY;  // smallest distance from a threshold
                {
                    float h[kB];
#pragma unroll
                    for (int j = 0; j < kB; ++j) h[j] = hb[j * HP + lb];
                    // thresholds and couplings are read two decisions ahead, one where
                    // the fields leave few registers
                    constexpr int kAhead = MS * KS > 32 ? 1 : 2;
                    float tn[kAhead];
                    f4 Jn[kAhead][4];
#pragma unroll
                    for (int z = 0; z < kAhead; ++z) {
                        tn[z] = tb[z * WP + lb];
#pragma unroll
                        for (int y = 0; y < 4; ++y) Jn[z][y] = J[4 * z + y];
                    }
                    // (a last block's places past N have no couplings; they are masked below)
                    static_for<0, kB>([&](auto JC) __attribute__((always_inline)) {
                        constexpr int j = decltype(JC)::value;
                        constexpr int o = j % kAhead;
                        const float thr = tn[o];
                        const f4 J0 = Jn[o][0], J1 = Jn[o][1], J2 = Jn[o][2], J3 = Jn[o][3];
                        const float Jr[kB] = {J0.x, J0.y, J0.z, J0.w, J1.x, J1.y, J1.z, J1.w,
                                              J2.x, J2.y, J2.z, J2.w, J3.x, J3.y, J3.z, J3.w};
                        if constexpr (j + kAhead < kB) {
                            tn[o] = tb[(j + kAhead) * WP + lb];
#pragma unroll
                            for (int y = 0; y < 4; ++y)
                                if (4 * y + 3 > j + kAhead) Jn[o][y] = J[(j + kAhead) * 4 + y];
                        }
                        const uint32_t sg = sb << (31 - j);  // sign bit: s = -1
                        const float d = __uint_as_float(flip_sign(__float_as_uint(h[j]), sg)) - thr;
                        dmin = fminf(dmin, fabsf(d));
                        // accepted below the threshold: d's sign bit
                        ab = __builtin_amdgcn_alignbit(ab, __float_as_uint(d), 31);
                        // the spin's change over 2
                        const uint32_t in = (uint32_t)((int32_t)__float_as_uint(d) >> 31);
                        const float ch = __uint_as_float(flip_sign(0xBF800000u, sg) & in);
#pragma unroll
                        for (int j2 = j + 1; j2 < kB; ++j2) h[j2] = __builtin_fmaf(ch, Jr[j2], h[j2]);
                        __builtin_amdgcn_sched_barrier(0);
                    });
                    ab = __brev(ab) >> 16;
                }
                // open spins, or no finite thresholds (NaN, which fminf passes over)
                const bool redo = __ballot(act && !(dmin > gd)) || !finite(T, jp);
                if (redo) {
                    // rare: the same in a loop, with the open spins' fields in double
                    const double jpd = (double)jp;
                    const int ml = tau == 0 ? (lb == 0 ? W - 1 : lb - 1) : lb;
                    const int mr = tau == 0 ? lb : (lb == W - 1 ? 0 : lb + 1);
                    float h[kB];
#pragma unroll
                    for (int j = 0; j < kB; ++j) h[j] = hb[j * HP + lb];
                    ab = 0;
#pragma unroll 1
                    for (int j = 0; j < nq; ++j) {
                        const int q = c * kB + j;
                        const WT S_ = mine[q], O = other[q];
                        const uint32_t sg = (uint32_t)(S_ >> lb) << 31;
                        const float thr = tb[j * WP + lb];
                        const float d = __uint_as_float(__float_as_uint(h[0]) ^ sg) - thr;
                        bool acc = d < -gd;
                        for (unsigned long long todo = __ballot(act && !acc && !(d > gd)); todo; todo &= todo - 1) {
                            const int lo = __ffsll(todo) - 1;  // slice whose field is summed, spins over the lanes
                            double e = 0.0;
#pragma unroll
                            for (int k = 0; k < KS; ++k) {
                                const int p = 64 * k + ln;
                                const float v = p < N ? a.j2[((size_t)q * 64 + ln) * KS + k] : 0.0f;
                                e += (p < N && ((mine[p] >> lo) & 1)) ? -(double)v : (double)v;
                            }
#pragma unroll
                            for (int o = 32; o > 0; o >>= 1) e += __shfl_xor(e, o, 64);
                            if (ln == lo) {
                                const double hx = 0.5 * e + a.diag[q];
                                const double ts = (((O >> ml) & 1) ? -1.0 : 1.0) + (((O >> mr) & 1) ? -1.0 : 1.0);
                                const double ed = -2.0 * (sg ? -1.0 : 1.0) * (hx + jpd * ts);
                                unsigned int tr = 0;
                                const int cls = piqmc_fixed_class(ed, (double)T, &tr);
                                acc = cls == 1 || (cls == 2 && uu[(buf * kB + j) * WP + lb] < tr);
                            }
                        }
                        const float ch = acc ? __uint_as_float(0xBF800000u ^ sg) : 0.0f;
                        const float *Jr = jb + (buf * kB + j) * kB;
#pragma unroll
                        for (int y = 0; y + 1 < kB; ++y) h[y] = __builtin_fmaf(ch, j + 1 + y < kB ? Jr[j + 1 + y] : 0.0f, h[y + 1]);
                        const WT F = (WT)__ballot(acc && act);
                        ab |= acc ? 1u << j : 0u;
                        // the sums above read the block's spins as decided so far
                        if (ln == 0) mine[q] = S_ ^ F;
                        wave_sync();
                    }
                }
                ab = act ? ab & ((1u << max(nq, 0)) - 1u) : 0u;
                const uint32_t flips = transpose32(ab, ln & 31);
                if (act) fm[ln] = ab | (sb << 16);
                if (holds) *half = old ^ flips;
                __builtin_amdgcn_s_setprio(0);
            } else if (on) {
                // this block's rows for the updates, the next block's couplings and draws
                // (straight to LDS, a wavefront's 64 groups at a time; groups past
                // the block's rows repeat its last one)
                const f4 *src = reinterpret_cast<const f4 *>(a.j2 + (size_t)c * kB * 64 * KS);
                const int last = nq * kV - 1;  // (below 0 in the empty block of a single one)
                for (int y = tw - 1; y < kB * kV / 64 && last >= 0; y += kTeam - 1)
                    __builtin_amdgcn_global_load_lds(
                        (const __attribute__((address_space(1))) void *)(src + min(y * 64 + lane, last)),
                        (__attribute__((address_space(3))) void *)(rows + y * 256), 16, 0, 0);
                if (more) {
                    if (tw == 1) stage_jb(cn, buf ^ 1);
                    for (int task = kTeam - 1 - tw; task < kTasks; task += kTeam - 1)
                        draw(task, cn, a.sweep_base + (uint32_t)(sn * a.M + mn), Tn, finite(Tn, jpn), buf ^ 1);
                }
                __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): the rows are in LDS before the barrier
            }
            __syncthreads();
            if (on) {
                // apply the block's flips to this wavefront's slices
                const uint32_t fv = fm[min(s0 + (lane & (MS - 1)), WP - 1)];
#pragma unroll
                for (int q = 0; q < MS; ++q) {
                    const uint32_t fs = q < ns ? (uint32_t)__builtin_amdgcn_readlane((int)fv, q) : 0u;
                    // two flips at a time (the second may be none)
                    for (uint32_t todo = fs & 0xffffu; todo;) {
                        const int j = __ffs(todo) - 1;
                        todo &= todo - 1;
                        const int i = todo ? __ffs(todo) - 1 : j;
                        const double sj = (fs >> (16 + j)) & 1u ? 1.0 : -1.0;  // -1 to +1 adds 2 J
                        const double si = todo ? ((fs >> (16 + i)) & 1u ? 1.0 : -1.0) : 0.0;
                        todo &= todo - 1;
                        float rj[KS], ri[KS];
#pragma unroll
                        for (int k = 0; k < KS; ++k) {
                            rj[k] = rows[(j * 64 + lane) * KS + k];
                            ri[k] = rows[(i * 64 + lane) * KS + k];
                        }
#pragma unroll
                        for (int k = 0; k < KS; ++k) f[q][k] = fma(si, (double)ri[k], fma(sj, (double)rj[k], f[q][k]));
                    }
                }
                if (more) hand_over(cn, jpn);
                c = cn;
                m = mn;
                s = more ? sn : s;
                T = Tn;
                jp = jpn;
                ++x;
                buf ^= 1;
            } else if (t == 0) {
                hand_over(c, jp);  // the odd team's first block
            }
            __syncthreads();
        }
        if (a.etrace) {
            // sum over slices of the classical energy: -(f + h) s / 2 per spin
            double e = 0.0;
#pragma unroll
            for (int k = 0; k < KS; ++k) {
                const int q = 64 * k + lane;
                if (q >= N) continue;
                const double dg = a.diag[q];
                const WT w = mine[q];
#pragma unroll
                for (int q2 = 0; q2 < MS; ++q2)
                    if (q2 < ns) {
                        const double v = 0.5 * (f[q2][k] + dg);
                        e -= ((w >> (s0 + q2)) & 1) ? -v : v;
                    }
            }
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) e += __shfl_xor(e, o, 64);
            if (lane == 0) red[wv] = e;
            __syncthreads();
            if (tid == 0) {
                double v = 0.0;
                for (int w = 0; w < 2 * kTeam; ++w) v += red[w];
                a.etrace[(size_t)r * a.S + seg] = v / (double)a.P;
            }
            __syncthreads();
        }
    }
    for (int y = tid; y < 2 * NP; y += blockDim.x) {
        const int q = y % NP;
        if (q < N) gst[(size_t)(y / NP) * N + a.order[q]] = st[y];
    }
}

template <typename WT, int KS>
__global__ void __launch_bounds__(128 * kTeam) block_kernel(BlockArgs a)
{
    extern __shared__ __align__(16) unsigned char smem[];
    block_sweep<WT, KS>(a, blockIdx.x, smem);
}

// Replicas of a batch's jobs from a device counter, longest first: resident
// workgroups leave once the counter has passed the items.
template <typename WT>
__device__ void block_item(const BlockArgs &a, int r, unsigned char *smem)
{
    switch ((a.N + 63) / 64) {
    case 1: block_sweep<WT, 1>(a, r, smem); break;
    case 2: block_sweep<WT, 2>(a, r, smem); break;
    case 3: block_sweep<WT, 3>(a, r, smem); break;
    default: block_sweep<WT, 4>(a, r, smem); break;
    }
}
__global__ void __launch_bounds__(128 * kTeam) batch_block_kernel(const BlockArgs *jobs, const int2 *items, int n, int *head)
{
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ int cur;
    for (;;) {
        __syncthreads();
        if (threadIdx.x == 0) cur = atomicAdd(head, 1);
        __syncthreads();
        const int it = __builtin_amdgcn_readfirstlane(cur);
        if (it >= n) break;
        const int2 item = items[it];
        const BlockArgs &a = jobs[__builtin_amdgcn_readfirstlane(item.x)];
        const int r = __builtin_amdgcn_readfirstlane(item.y);
        if (a.W <= 32) block_item<uint32_t>(a, r, smem);
        else block_item<uint64_t>(a, r, smem);
    }
}

template <typename WT, int KS>
int launch(const BlockArgs &a, hipStream_t st)
{
    const size_t lds = block_lds(a.N, sizeof(WT));
    PIQMC_HIP(hipFuncSetAttribute((const void *)block_kernel<WT, KS>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    block_kernel<WT, KS><<<a.R, 128 * kTeam, lds, st>>>(a);
    PIQMC_HIP(hipGetLastError());
    return PIQMC_OK;
}

template <typename WT>
int launch_slots(const BlockArgs &a, hipStream_t st)
{
    switch ((a.N + 63) / 64) {
    case 1: return launch<WT, 1>(a, st);
    case 2: return launch<WT, 2>(a, st);
    case 3: return launch<WT, 3>(a, st);
    default: return launch<WT, 4>(a, st);
    }
}

}  // namespace

namespace piqmc {

BlockArgs block_args(const piqmc_problem *p)
{
    BlockArgs a = {};
    a.N = p->N;
    a.order = p->d_order;
    const int slots = (p->N + 63) / 64;
    a.diag = reinterpret_cast<const double *>(p->d_block);
    a.j2 = reinterpret_cast<const float *>(p->d_block + sizeof(double) * 64 * slots);
    a.jb2 = a.j2 + (size_t)p->N * 64 * slots;
    a.bound = p->block_bound;
    return a;
}

int block_launch(const BlockArgs &a, hipStream_t st)
{
    return a.W <= 32 ? launch_slots<uint32_t>(a, st) : launch_slots<uint64_t>(a, st);
}

size_t block_item_lds(const BlockArgs &a) { return block_lds(a.N, a.W <= 32 ? 4 : 8); }

int block_batch_prepare(size_t lds)
{
    PIQMC_HIP(hipFuncSetAttribute((const void *)batch_block_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    return PIQMC_OK;
}

void block_batch_launch(const BlockArgs *jobs, const int2 *items, int n, int *head, int grid, size_t lds, hipStream_t st)
{
    batch_block_kernel<<<grid, 128 * kTeam, lds, st>>>(jobs, items, n, head);
}

// [diag | twice the couplings | those within blocks] by color position, where the blocked sweep
// applies: every row exact in any order and symmetric, color classes of fewer
// than 8 spins on average (else a word per thread is the faster layout), no
// coupling that doubling would overflow.
int block_upload(piqmc_problem &p, const std::vector<int32_t> &order)
{
    if (p.d_block) (void)hipFree(p.d_block);
    p.d_block = nullptr;
    const int N = p.N, slots = (N + 63) / 64;
    if (N > kBlockMaxN || !p.exact_rows || !p.fields_ok || N >= 8 * p.ncolors) return PIQMC_OK;
    std::vector<int> pos(N);
    for (int q = 0; q < N; ++q) pos[order[q]] = q;
    const size_t bd = sizeof(double) * 64 * slots;
    const int nb = (N + kB - 1) / kB;
    std::vector<unsigned char> img(bd + sizeof(float) * ((size_t)N * 64 * slots + (size_t)nb * kB * kB), 0);
    double *diag = reinterpret_cast<double *>(img.data());
    float *j2 = reinterpret_cast<float *>(img.data() + bd), *jb2 = j2 + (size_t)N * 64 * slots;
    double bound = 0.0;
    for (int i = 0; i < N; ++i) {
        double sum = 0.0;
        for (int e = 0; e < p.Z; ++e) {
            const float J = p.J[(size_t)i * p.Z + e];
            const int j = p.idx[(size_t)i * p.Z + e];
            if (J == 0.0f) continue;
            sum += fabs((double)J);
            if (j == i) diag[pos[i]] += (double)J;
            else {
                const int q = pos[i], k = pos[j];
                j2[((size_t)q * 64 + (k & 63)) * slots + (k >> 6)] = 2.0f * J;
                if (q / kB == k / kB) jb2[((size_t)(q / kB) * kB + q % kB) * kB + k % kB] = 2.0f * J;
            }
        }
        bound = std::max(bound, sum);
    }
    if (!(bound < 1e30)) return PIQMC_OK;
    p.block_bound = (float)(bound * 1.000001);
    PIQMC_HIP(hipMalloc((void **)&p.d_block, img.size()));
    PIQMC_HIP(hipMemcpy(p.d_block, img.data(), img.size(), hipMemcpyHostToDevice));
    return PIQMC_OK;
}

}  // namespace piqmc
