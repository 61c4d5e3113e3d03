// rki4 summary build for gfx950: finalized K pages -> six-slab summaries.
//
// Op sequence of the reference builder (selection/rki4_build.py:147-158
// _write_pre, :93-129 eigh, :178-225 _write_post, :161-175 int4 pack), per
// (block, kv head):
//   mu = mean_t K; dc = K - mu; Gm = dc dc^T (16 x 16)
//   S2, U = eigh(Gm) ascending; S8 = sqrt(max(S2[-8:], 1e-10)); U8 = U[:, -8:]
//   C = U8 * S8 ; V = dc^T U8 / S8
//   vs = max(|V|_d / 7, 1e-8);  Vq = clamp(rint(V / vs), -8, 7)  -> int4 packed
//   cs = max(|C|_r / 127, 1e-8); Cq = clamp(rint(C / cs), +-127)
//   ms = max(|mu| / 127, 1e-8); muq = clamp(rint(mu / ms), +-127)
//   scales stored bf16 (RNE); tag = K[15, kh, 0:8].
//
// MI355X mapping: a wave builds up to 64 / page pages at once, a page on `page`
// lanes, with the gram and the eigenvectors in registers (rki4_build_kernel).
// The gram runs on v_mfma_f32_16x16x4_f32 (A and B operands are the same lane
// values because Gm = dc dc^T); the eigendecomposition is a parallel cyclic
// Jacobi (round-robin ordering: page / 2 disjoint rotations per step, page - 1
// steps per sweep) -- the reference calls a batched LAPACK/cuSOLVER eigh; any
// eigensolver agrees with it only up to eigenvector sign/rotation, which the
// summary tolerates by design.  locks_pack_rki4 takes the eigenpairs from the
// caller and follows the reference's op order (V accumulated over t in
// ascending order, IEEE division, round-half-even), which the build shares.
#include <algorithm>
#include <type_traits>

#include "locks_common.h"
#include "locks_hip.h"

namespace locks {

constexpr int BD_RNK = 8;
// build grid cap (waves stride over the rest): a few resident rounds on 256 CUs
constexpr long BD_MAX_GRID = 4096;
// waves that the items are spread over before a wave takes another page (up to
// 64 / page): one per SIMD of the chip.  1024 pages 60 us at one a wave; 1600
// pages 63 us at two (70 at four), 2400 68 us at three (70), 4096 72 us at four
constexpr long BD_SPREAD = 1024;
// pages per wave, at most gw (1, 2 or 4), of `items` on `waves` waves.  The host
// sizes the grid with it for the bound that it knows; the kernel packs what the
// device count says (8 layers, 4 blocks to build of a bound of 2048, packed by
// the bound / by the count: d 512 89 / 58 us, 8 heads of d 128 58 / 49).
__host__ __device__ __forceinline__ int pages_per_wave(long items, long waves, int gw) {
    const long n = waves < BD_SPREAD ? waves : BD_SPREAD;
    int g = 1;
    for (int k = 1; k < gw; ++k) g += items > k * n ? 1 : 0;
    return g;
}

__device__ __forceinline__ long readlane64(long v, int l) {
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)v, l), hi = (uint32_t)__builtin_amdgcn_readlane((int)(v >> 32), l);
    return (long)(((uint64_t)hi << 32) | lo);
}
// value of another lane; addr = 4 x lane
__device__ __forceinline__ float from_lane(int addr, float v) {
    return __int_as_float(__builtin_amdgcn_ds_bpermute(addr, __float_as_int(v)));
}
// a in the lanes of mask m, b in the others.  Selects are spelled by mask: as
// conditionals on a lane's own index the compiler makes the row array an
// indexed one, in scratch memory.
__device__ __forceinline__ float pick(uint64_t m, float a, float b) {
    return __builtin_amdgcn_inverse_ballot_w64(m) ? a : b;
}
// a in lane I of every page, b elsewhere.  The mask is made where it is used
// (scalar moves): as plain constants the masks of all I are hoisted together
// and spilled to VGPR lanes, a read each.
template <int N, int I>
__device__ __forceinline__ float pick_lane(float a, float b) {
    constexpr uint64_t M = (N == 16 ? 0x0001000100010001ull : N == 32 ? 0x0000000100000001ull : 1ull) << I;
    uint32_t lo, hi;
    asm volatile("s_mov_b32 %0, %1" : "=s"(lo) : "i"((int)(uint32_t)M));
    if constexpr ((uint32_t)(M >> 32) == (uint32_t)M) hi = lo;
    else asm volatile("s_mov_b32 %0, %1" : "=s"(hi) : "i"((int)(uint32_t)(M >> 32)));
    return pick(((uint64_t)hi << 32) | lo, a, b);
}
template <int B, int E, class F>
__device__ __forceinline__ void static_for(F&& f) {
    if constexpr (B < E) {
        f(std::integral_constant<int, B>{});
        static_for<B + 1, E>(f);
    }
}
// sum over the N lanes of a page, result in each
template <int N>
__device__ __forceinline__ float lanes_sum(float v) {
    v += row_ror<8>(v);
    v += row_ror<4>(v);
    v += row_ror<2>(v);
    v += row_ror<1>(v);
    if constexpr (N >= 32) v = xor16_sum(v);
    if constexpr (N >= 64) v = xor32_sum(v);
    return v;
}

// ---- build ------------------------------------------------------------------
// One wave builds up to 64 / PG pages at once: a page of PG tokens is PG
// lanes, and lane j holds column j of the page's gram and row j of its
// eigenvectors in registers (2 PG VGPRs), so the row half of a Jacobi rotation
// is register arithmetic and only the gram's column half moves data between
// lanes (PG ds_bpermute per step, no LDS storage).  With one page per wave and
// both matrices in LDS the build was bound by its LDS accesses (page 16: ~47
// per step and page) and, one page alone, by their latency.  The rotations round
// as they did; the stop test sums in another order, so a page right at its bound
// may take a sweep more or less (none of the pages compared did: bytes equal).
// Measured, before -> after:
//   8 layers x 2048 pages x 8 heads, d 128 page 16   4.06 -> 0.92 ms (7.0 ns a page)
//   8 layers x 2048 latent pages, d 512              1.20 -> 0.26 ms
//   4 layers x 512 pages x 8 heads, d 128 page 32    6.52 -> 0.96 ms
//   4 layers x 256 pages x 8 heads, d 128 page 64    135 -> 3.85 ms
//   32 layers x 8 heads x 4 pages (one a wave)       82 -> 58 us
// What bounds page 16 now: the Jacobi takes 2/3 of the time, ~120 clocks per CU
// for a wave's step of ~140-167 VALU instructions and 23 LDS operations (18
// exchanges), four waves a SIMD.  Both pipes are near full: the schedule from a
// table instead of arithmetic (27 VALU instructions fewer a step) gave 1 %, and
// made a lone page slower (57 -> 61 us, its scalar loads wait).  The gram, the
// pack and their loads are the rest.

// Parallel cyclic Jacobi, round-robin ordering: index 0 stays, 1 .. N - 1
// rotate.  At step s index i > 0 sits in slot 1 + (i - 1 - s) mod (N - 1);
// slot 0 (index 0) pairs with slot 1, slot m > 1 with slot N + 1 - m; a pair is
// (p, q) with p in slot 0 or 2 .. N / 2.  Rows are kept in slot order: a step
// writes each row one slot down, so every step is the same code.  One step
// applies the N / 2 disjoint rotations as A'' = J^T A J from the old A:
//   A''[i][j] = c_j (c_i A[i][j] + s_i A[pi][j]) + s_j (c_i A[i][pj] + s_i A[pi][pj])
//   U'[i][j]  = c_j U[i][j] + s_j U[i][pj]
// A is kept by columns (lane j: column j), U by rows (lane t: row t, its
// columns in slot order too), so only A's column half needs an exchange.
// Rotation parameters use the hardware reciprocal and reciprocal square root
// (~1 ulp): a rotation only has to reduce the off-diagonal mass, and the
// result is checked through the quantised summary, not bit for bit.
// `cs`: this page's N / 2 (c, s) pairs in LDS.  On return `diag` is the
// eigenvalue of column j = lane % N and U the eigenvectors' entries of token j.
template <int N>
__device__ __forceinline__ void jacobi(float (&A)[N], float (&U)[N], float& diag, float2* cs, int lane) {
    static_assert(N == 16 || N == 32 || N == 64, "page 16, 32 or 64");
    constexpr int SWEEPS = N == 16 ? 12 : N == 32 ? 16 : 20;
    const int base = lane & ~(N - 1);
    bool done = false;
#pragma unroll 1
    for (int sweep = 0; sweep < SWEEPS; ++sweep) {
        // Off-diagonal mass against the diagonal, per page (also done on 0/0).
        // fp32 rounding leaves off/dia near 1e-14 (asymmetric residues of
        // order eps * |lambda|), so the bound sits above that floor: 5-6 sweeps
        // at N = 16 instead of running out the sweep limit, with the same top-8
        // eigenvalue accuracy (~3e-6 rel).
        float off = 0.f, dia = diag * diag;
        static_for<0, N>([&](auto ic) {
            constexpr int i = decltype(ic)::value;
            const float a = pick_lane<N, i>(0.f, A[i]);
            off = __builtin_fmaf(a, a, off);
        });
        off = lanes_sum<N>(off);
        dia = lanes_sum<N>(dia);
        done = done || !(off > 1e-12f * dia);
        if (__ballot(!done) == 0) break;
        int slot = lane & (N - 1);
        // (three steps a turn where they divide the sweep: results then land
        // in their registers without moves)
#pragma unroll N == 32 ? 1 : 3
        for (int step = 0; step < N - 1; ++step) {
            const int ps = slot < 2 ? 1 - slot : N + 1 - slot;       // the partner's slot and lane
            int pi = ps + step;
            pi = pi >= N ? pi - (N - 1) : pi;
            pi = ps == 0 ? 0 : pi;
            const int addr = (base | pi) << 2;
            const float pd = from_lane(addr, diag);
            // this column's element in the partner's row
            float t[N / 2];
            const uint64_t odd = __ballot(ps & 1);
#pragma unroll
            for (int i = 0; i < N / 2; ++i) t[i] = pick(odd, A[2 * i + 1], A[2 * i]);
#pragma unroll
            for (int b = 2, n = N / 4; n >= 1; b *= 2, n /= 2) {
                const uint64_t m = __ballot(ps & b);
#pragma unroll
                for (int i = 0; i < n; ++i) t[i] = pick(m, t[2 * i + 1], t[2 * i]);
            }
            const float po = from_lane(addr, t[0]);
            // first of its pair (p): slot 0 or 2 .. N / 2
            const uint64_t first = __ballot(((slot == 0) | ((unsigned)(slot - 2) <= (unsigned)(N / 2 - 2))) != 0);
            const float sgn = pick(first, 1.f, -1.f);
            const float apq = pick(first, po, t[0]);                 // A[p][q] is column q's
            // A[q][q] - A[p][p], the same on both lanes down to the zero's sign
            const float theta = __builtin_fmaf(pd, sgn, -(diag * sgn)) * __builtin_amdgcn_rcpf(2.f * apq);
            const float tt = copysignf(__builtin_amdgcn_rcpf(fabsf(theta) +
                                                             __builtin_amdgcn_sqrtf(__builtin_fmaf(theta, theta, 1.f))),
                                       theta);
            const float cr = __builtin_amdgcn_rsqf(__builtin_fmaf(tt, tt, 1.f));
            const bool rot = !done && fabsf(apq) > 1e-30f;           // smaller: nothing to rotate away
            const float c = rot ? cr : 1.f, sn = rot ? tt * cr : 0.f;
            const float sj = -sgn * sn;
            const int e = min(slot, ps);                             // the pair's place: p's slot, 0 and 2 .. N / 2
            cs[e == 0 ? 0 : e - 1] = make_float2(c, sn);             // (both lanes of the pair: the same value)
            asm volatile("" ::: "memory");
            // the diagonal element, with the roundings of the full update
            const float d0 = __builtin_fmaf(c, diag, sj * t[0]), d1 = __builtin_fmaf(c, po, sj * pd);
            const float nd = __builtin_fmaf(c, d0, sj * d1);
            diag = done ? diag : nd;
            float B[N], W[N];
#pragma unroll
            for (int k = 0; k < N / 2; ++k) {
                const float2 r = cs[k];
                const int p = k == 0 ? 0 : k + 1, q = k == 0 ? 1 : N - k;
                B[p] = __builtin_fmaf(r.x, A[p], -(r.y * A[q]));
                B[q] = __builtin_fmaf(r.x, A[q], r.y * A[p]);
                W[p] = __builtin_fmaf(r.x, U[p], -(r.y * U[q]));
                W[q] = __builtin_fmaf(r.x, U[q], r.y * U[p]);
            }
            asm volatile("" ::: "memory");
            // (issued together: left to the scheduler each exchange is waited
            // for before the next goes out, 82 -> 72 us for 1024 single pages)
            float pb[N];
#pragma unroll
            for (int i = 0; i < N; ++i) pb[i] = from_lane(addr, B[i]);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < N; ++i)
                A[i == 0 ? 0 : i == 1 ? N - 1 : i - 1] = __builtin_fmaf(c, B[i], sj * pb[i]);
#pragma unroll
            for (int i = 0; i < N; ++i) U[i == 0 ? 0 : i == 1 ? N - 1 : i - 1] = W[i];
            slot = slot < 2 ? (slot == 0 ? 0 : N - 1) : slot - 1;
        }
    }
}

// a / b, correctly rounded, from y = RN(1 / b): the quotient estimate a y and
// one residual correction (Markstein 1990; exact away from under- / overflow:
// scales are at least 1e-8, so what underflows is a zero code either way).
// b infinite (a page with infinite keys, or an overflowing gram): y is 0 and
// the residual is taken against br = 0 in place of b, so a finite a gives 0
// and not NaN.
__device__ __forceinline__ float residual_divisor(float b, float y) { return y == 0.f ? 0.f : b; }
__device__ __forceinline__ float div_by(float a, float br, float y) {
    const float q = a * y;
    return __builtin_fmaf(__builtin_fmaf(-q, br, a), y, q);
}

typedef const __attribute__((address_space(1))) uint32_t* global_u32;

// Per-wave LDS: a window of one page's centred channels for the gram (pitch a
// multiple of 4 words that is odd in quads, so the operand reads spread over
// all banks), then the rotation pairs, then the kept columns of every page
// with their singular values and reciprocals.
template <int PG>
struct BuildLds {
    static constexpr int GW = kWave / PG;            // pages per wave
    static constexpr int WIN = 128 * 16 / PG;        // channels per window
    union {
        float dc[PG][WIN + 4];
        float2 cs[GW][PG / 2];
        struct {
            float u[GW][BD_RNK][PG];
            float s8[GW][BD_RNK], r8[GW][BD_RNK], y8[GW][BD_RNK];    // values, residual divisors, reciprocals
            uint32_t lam[kWave];
        } top;
    };
};

// One wave takes gpw (1 to 64 / PG) consecutive (layer, block, kv head) items at a
// time, and waves stride over the rest.  Layer l reads K from k_layers[l] (or kc
// for a single-layer call) and writes slab rows offset by l * layer_rows.
// n_dev, when given, is a device count of valid entries of `blocks` (at most
// n_blocks): the refresh producers size the grid to the host-known bound and
// the list is compacted on the device.
template <int D, int PG>
__global__ __launch_bounds__(256, PG == 16 && D <= 128 ? 4 : 2) void rki4_build_kernel(
    const uint16_t* __restrict__ kc, const uint64_t* __restrict__ k_layers,
    long k_sb, long k_st, long k_sh, int NB,
    const int* __restrict__ blocks, const int* __restrict__ n_dev, int n_blocks, int n_kv,
    int n_layers, long layer_rows, SlabRows S, uint16_t* __restrict__ tag)
{
    using LDS = BuildLds<PG>;
    constexpr int NW = 4, GW = LDS::GW, NB16 = PG / 16;
    constexpr int LPP = D >= 128 ? 64 : D / 2;       // lanes that share a page's channels
    constexpr int NK = D >= 128 ? D / 128 : 1;       // 128-channel groups; lane l: channels 2 l, 2 l + 1 of each
    constexpr int WIN = LDS::WIN, WCH = D < WIN ? D : WIN, NWIN = (D < 128 ? D : 128) / WCH;
    __shared__ __attribute__((aligned(16))) LDS lds[NW];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    LDS& L = lds[wave];
    const int nb_valid = n_dev ? min(*n_dev, n_blocks) : n_blocks;
    const long per_layer = (long)nb_valid * n_kv, total = per_layer * n_layers;
    const int gpw = pages_per_wave(total, (long)gridDim.x * NW, GW);
    const int j = lane & (PG - 1), pg = lane / PG;   // this lane's column / token, and page
    const bool own = lane < LPP;                     // d = 64: the upper lanes repeat, and store nothing
    const int cl = own ? lane : lane - LPP;
    for (long base = ((long)blockIdx.x * NW + wave) * gpw; base < total; base += (long)gridDim.x * NW * gpw) {
        // this lane's page: K address (null: none) and summary row
        const uint16_t* kpl = nullptr;
        long rwl = 0;
        if (pg < gpw && base + pg < total) {
            const long it = base + pg;
            const int layer = total <= 0xFFFFFFFFL ? (int)((uint32_t)it / (uint32_t)per_layer) : (int)(it / per_layer);
            const uint32_t rem = (uint32_t)(it - (long)layer * per_layer);      // < n_blocks * n_kv
            const uint32_t bi = rem / (uint32_t)n_kv;
            const int blk = blocks[bi];
            if (blk >= 0 && blk < NB) {                                // else masked (profile pass)
                const int kh = (int)(rem - bi * (uint32_t)n_kv);
                rwl = (long)layer * layer_rows + (long)blk * n_kv + kh;
                kpl = (k_layers ? reinterpret_cast<const uint16_t*>(k_layers[layer]) : kc) +
                      (long)blk * k_sb + (long)kh * k_sh;
            }
        }
        // the same of page g of the wave, wave-uniform
        auto page_row = [&](int g) { return readlane64(rwl, g * PG); };
        auto page_k = [&](int g) { return reinterpret_cast<const uint16_t*>(readlane64(reinterpret_cast<long>(kpl), g * PG)); };
        // the page's tokens of channels 2 l, 2 l + 1 of group k, minus their
        // mean (a sequential sum over t; 1 / PG is a power of two)
        auto centred = [&](const uint16_t* p, int k, float (&x)[PG][2], float (&mu)[2]) {
            uint32_t w[PG];
#pragma unroll
            for (int t = 0; t < PG; ++t) w[t] = ((global_u32)(p + (long)t * k_st + 128 * k))[cl];
            float a = 0.f, b = 0.f;
#pragma unroll
            for (int t = 0; t < PG; ++t) { a = __fadd_rn(a, bf16lo(w[t])); b = __fadd_rn(b, bf16hi(w[t])); }
            mu[0] = __fmul_rn(a, 1.f / PG);
            mu[1] = __fmul_rn(b, 1.f / PG);
#pragma unroll
            for (int t = 0; t < PG; ++t) {
                x[t][0] = __fsub_rn(bf16lo(w[t]), mu[0]);
                x[t][1] = __fsub_rn(bf16hi(w[t]), mu[1]);
            }
        };

        // ---- gram on the matrix core, Gm[i][j] = sum_d dc[i][d] dc[j][d], one
        // page after the other, in 16 x 16 blocks (bi, bj)
        const int i16 = lane & 15, kq = lane >> 4;
        v4f gm[GW][NB16][NB16];
#pragma unroll
        for (int g = 0; g < GW; ++g) {
#pragma unroll
            for (int bi = 0; bi < NB16; ++bi)
#pragma unroll
                for (int bj = 0; bj < NB16; ++bj) gm[g][bi][bj] = v4f{0.f, 0.f, 0.f, 0.f};
            const uint16_t* kp = page_k(g);
            if (kp == nullptr) continue;
#pragma unroll 1
            for (int k = 0; k < NK; ++k) {
                float x[PG][2], mu[2];
                centred(kp, k, x, mu);
#pragma unroll 1
                for (int wi = 0; wi < NWIN; ++wi) {
                    const int at = 2 * lane - WCH * wi;
                    if (at >= 0 && at < WCH)
#pragma unroll
                        for (int t = 0; t < PG; ++t)
                            *reinterpret_cast<float2*>(&L.dc[t][at]) = make_float2(x[t][0], x[t][1]);
                    wave_lds_sync();
#pragma unroll 4
                    for (int s = 0; s < WCH / 4; ++s) {
                        float a[NB16];
#pragma unroll
                        for (int bi = 0; bi < NB16; ++bi) a[bi] = L.dc[16 * bi + i16][4 * s + kq];
#pragma unroll
                        for (int bi = 0; bi < NB16; ++bi)
#pragma unroll
                            for (int bj = 0; bj < NB16; ++bj)
                                gm[g][bi][bj] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[bi], a[bj], gm[g][bi][bj], 0, 0, 0);
                    }
                    wave_lds_sync();
                }
            }
        }
        // lane (kq, i) holds rows 4 kq .. 4 kq + 3 of column i of each block;
        // exchange so that each lane holds all PG rows of its own column
        float A[PG], U[PG], diag = 0.f;
#pragma unroll
        for (int bi = 0; bi < NB16; ++bi)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                uint32_t r[4];
#pragma unroll
                for (int x = 0; x < 4; ++x) r[x] = __float_as_uint(gm[x / NB16][bi][x % NB16][v]);
                const auto s02 = __builtin_amdgcn_permlane32_swap(r[0], r[2], false, false);
                const auto s13 = __builtin_amdgcn_permlane32_swap(r[1], r[3], false, false);
                const auto s01 = __builtin_amdgcn_permlane16_swap(s02[0], s13[0], false, false);
                const auto s23 = __builtin_amdgcn_permlane16_swap(s02[1], s13[1], false, false);
                A[16 * bi + v] = __uint_as_float(s01[0]);
                A[16 * bi + 4 + v] = __uint_as_float(s01[1]);
                A[16 * bi + 8 + v] = __uint_as_float(s23[0]);
                A[16 * bi + 12 + v] = __uint_as_float(s23[1]);
            }
        static_for<0, PG>([&](auto ic) {
            constexpr int i = decltype(ic)::value;
            U[i] = pick_lane<PG, i>(1.f, 0.f);
            diag = pick_lane<PG, i>(A[i], diag);
        });
        jacobi<PG>(A, U, diag, L.cs[pg], lane);
        wave_lds_sync();
        // ---- ascending ranks; the 8 largest: columns, singular values --------
        {
            // order-preserving key; NaN (a page with non-finite keys) lowest, ties by column
            const uint32_t key = f2u(diag == diag ? diag + 0.f : -INFINITY);
            L.top.lam[lane] = key;
            wave_lds_sync();
            int rank = 0;
#pragma unroll
            for (int m = 0; m < PG; m += 4) {
                const uint4 l4 = *reinterpret_cast<const uint4*>(&L.top.lam[lane - j + m]);
                const uint32_t lk[4] = {l4.x, l4.y, l4.z, l4.w};
#pragma unroll
                for (int e = 0; e < 4; ++e) rank += lk[e] < key + ((uint32_t)(m + e - j) >> 31) ? 1 : 0;
            }
            if (rank >= PG - BD_RNK) {
                const int r = rank - (PG - BD_RNK);
                const float s8 = __fsqrt_rn(fmaxf(diag, 1e-10f));
                const float y8 = __fdiv_rn(1.f, s8);
                L.top.s8[pg][r] = s8;
                L.top.r8[pg][r] = residual_divisor(s8, y8);
                L.top.y8[pg][r] = y8;
            }
            L.top.lam[lane] = (uint32_t)rank;        // (every key has been read)
            wave_lds_sync();
#pragma unroll
            for (int m = 0; m < PG; m += 4) {
                const uint4 l4 = *reinterpret_cast<const uint4*>(&L.top.lam[lane - j + m]);
                const uint32_t lk[4] = {l4.x, l4.y, l4.z, l4.w};
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (lk[e] >= PG - BD_RNK) L.top.u[pg][lk[e] - (PG - BD_RNK)][j] = U[m + e];
            }
            wave_lds_sync();
        }
        // ---- coefficients: this lane owns token j of page pg ------------------
        {
            if (kpl != nullptr) {
                float C[BD_RNK], am = 0.f;
#pragma unroll
                for (int r = 0; r < BD_RNK; ++r) {
                    C[r] = __fmul_rn(L.top.u[pg][r][j], L.top.s8[pg][r]);
                    am = fmaxf(am, fabsf(C[r]));
                }
                const float csc = fmaxf(__fdiv_rn(am, 127.f), 1e-8f), y = __fdiv_rn(1.f, csc), cr = residual_divisor(csc, y);
                uint32_t wd[2] = {0u, 0u};
#pragma unroll
                for (int r = 0; r < BD_RNK; ++r) {
                    const int q = (int)fminf(fmaxf(rintf(div_by(C[r], cr, y)), -127.f), 127.f);
                    wd[r >> 2] |= (uint32_t)(q & 255) << (8 * (r & 3));
                }
                *reinterpret_cast<uint2*>(S.c8 + rwl * S.sc8 + j * BD_RNK) = make_uint2(wd[0], wd[1]);
                reinterpret_cast<uint16_t*>(S.cs + rwl * S.scs)[j] = f32_to_bf16(csc);
                if (j < 8) tag[rwl * 8 + j] = kpl[(long)(PG - 1) * k_st + j];
            }
        }
        // ---- basis and centroid, one page after the other ---------------------
#pragma unroll 1
        for (int g = 0; g < gpw; ++g) {
            const uint16_t* kp = page_k(g);
            if (kp == nullptr) continue;
            const long rw = page_row(g);
            float V[NK][2][BD_RNK], mu[NK][2];
#pragma unroll
            for (int k = 0; k < NK; ++k) {
                float x[PG][2];
                centred(kp, k, x, mu[k]);
#pragma unroll
                for (int r = 0; r < BD_RNK; ++r) {
                    float a = 0.f, b = 0.f;                 // sequential over t
#pragma unroll
                    for (int t = 0; t < PG; ++t) {
                        const float u = L.top.u[g][r][t];
                        a = __fadd_rn(a, __fmul_rn(x[t][0], u));
                        b = __fadd_rn(b, __fmul_rn(x[t][1], u));
                    }
                    const float r8 = L.top.r8[g][r], y8 = L.top.y8[g][r];
                    V[k][0][r] = div_by(a, r8, y8);
                    V[k][1][r] = div_by(b, r8, y8);
                }
            }
            // Maxima over the channels of the 8 columns and the centroid.  Two
            // pair swaps fold the columns into one lane row each (lane row x of
            // m[0]: column x' = 2 (x & 1) + (x >> 1), of m[1]: 4 + x'), then each
            // row reduces; its lanes 0, 1, 2 turn the two columns' and the
            // centroid's maximum into a scale, read back lane by lane.
            float m[BD_RNK], mm = 0.f;
#pragma unroll
            for (int k = 0; k < NK; ++k) mm = fmaxf(mm, fmaxf(fabsf(mu[k][0]), fabsf(mu[k][1])));
            mm = wave_max(mm);
#pragma unroll
            for (int r = 0; r < BD_RNK; ++r) {
                m[r] = 0.f;
#pragma unroll
                for (int k = 0; k < NK; ++k) m[r] = fmaxf(m[r], fmaxf(fabsf(V[k][0][r]), fabsf(V[k][1][r])));
            }
#pragma unroll
            for (int r = 0; r < BD_RNK / 2; ++r) {            // columns 2 r (lower half), 2 r + 1
                const auto w = __builtin_amdgcn_permlane32_swap(__float_as_uint(m[2 * r]), __float_as_uint(m[2 * r + 1]), false, false);
                m[r] = fmaxf(__uint_as_float(w[0]), __uint_as_float(w[1]));
            }
#pragma unroll
            for (int r = 0; r < BD_RNK / 4; ++r) {
                const auto w = __builtin_amdgcn_permlane16_swap(__float_as_uint(m[2 * r]), __float_as_uint(m[2 * r + 1]), false, false);
                float x = fmaxf(__uint_as_float(w[0]), __uint_as_float(w[1]));
                x = fmaxf(x, row_ror<8>(x));
                x = fmaxf(x, row_ror<4>(x));
                x = fmaxf(x, row_ror<2>(x));
                m[r] = fmaxf(x, row_ror<1>(x));
            }
            const float am = i16 == 0 ? m[0] : i16 == 1 ? m[1] : mm;
            const float sc = fmaxf(__fdiv_rn(am, i16 < 2 ? 7.f : 127.f), 1e-8f);
            const float ys = __fdiv_rn(1.f, sc), sr = residual_divisor(sc, ys);
            if (i16 < 2)
                reinterpret_cast<uint16_t*>(S.vs + rw * S.svs)[4 * i16 + 2 * (kq & 1) + (kq >> 1)] = f32_to_bf16(sc);
            if (lane == 2) *reinterpret_cast<uint16_t*>(S.mus + rw * S.smus) = f32_to_bf16(sc);
            auto of_lane = [](float v, int l) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l)); };
            uint8_t* vrow = S.v4 + rw * S.sv4;
#pragma unroll
            for (int r = 0; r < BD_RNK; ++r) {
                const int at = 16 * (((r & 1) << 1) | ((r >> 1) & 1)) + (r >> 2);   // the lane of column r
                const float b = of_lane(sr, at), y = of_lane(ys, at);
#pragma unroll
                for (int k = 0; k < NK; ++k) {
                    const int lo = (int)fminf(fmaxf(rintf(div_by(V[k][0][r], b, y)), -8.f), 7.f);
                    const int hi = (int)fminf(fmaxf(rintf(div_by(V[k][1][r], b, y)), -8.f), 7.f);
                    if (own) vrow[r * (D / 2) + 64 * k + lane] = (uint8_t)((lo & 15) | ((hi & 15) << 4));
                }
            }
            const float b = of_lane(sr, 2), y = of_lane(ys, 2);
#pragma unroll
            for (int k = 0; k < NK; ++k) {
                const int lo = (int)fminf(fmaxf(rintf(div_by(mu[k][0], b, y)), -127.f), 127.f);
                const int hi = (int)fminf(fmaxf(rintf(div_by(mu[k][1], b, y)), -127.f), 127.f);
                if (own)
                    reinterpret_cast<uint16_t*>(S.mu + rw * S.smu)[64 * k + lane] =
                        (uint16_t)((lo & 255) | ((hi & 255) << 8));
            }
        }
        wave_lds_sync();                                     // the columns are read before the next gram
    }
}

// ---- locks_pack_rki4 ----------------------------------------------------------
// One page of PK_PG tokens x PK_D dims and the caller's eigenvectors, per wave.
constexpr int PK_D = 128, PK_PG = 16;
struct PackLds {
    float dc[PK_PG][PK_D + 1];   // centred page (padded rows)
    float mu[PK_D];
    float U[PK_PG][PK_PG + 1];   // eigenvectors (columns, ascending: the last 8 are kept)
    float S8[BD_RNK];
};

// quantize + pack one page, writing the six slab rows.  Lane l owns packed
// byte l of each column (d = 2 l, 2 l + 1).
__device__ __forceinline__ void pack_page(PackLds& L, long row, const SlabRows& S) {
    static_assert(PK_D == 2 * kWave, "two dims per lane");
    const int lane = threadIdx.x & 63;
    // V[d][r]: sequential over t, separately rounded
    float V[2][BD_RNK];
#pragma unroll
    for (int e = 0; e < 2; ++e)
#pragma unroll
        for (int r = 0; r < BD_RNK; ++r) {
            // a compiler barrier keeps one column's operands live at a time
            asm volatile("" ::: "memory");
            float acc = 0.f;
            for (int t = 0; t < PK_PG; ++t)
                acc = __fadd_rn(acc, __fmul_rn(L.dc[t][2 * lane + e], L.U[t][PK_PG - BD_RNK + r]));
            V[e][r] = __fdiv_rn(acc, L.S8[r]);
        }
    // per-column absmax over d (all of them before the first code: taken column by
    // column, the loads of every column move up and hold 480 VGPRs against 74)
    float vsc[BD_RNK];
#pragma unroll
    for (int r = 0; r < BD_RNK; ++r)
        vsc[r] = fmaxf(__fdiv_rn(wave_max(fmaxf(fabsf(V[0][r]), fabsf(V[1][r]))), 7.f), 1e-8f);
    uint8_t* vrow = S.v4 + row * S.sv4;
#pragma unroll
    for (int r = 0; r < BD_RNK; ++r) {
        const int lo = (int)fminf(fmaxf(rintf(__fdiv_rn(V[0][r], vsc[r])), -8.f), 7.f);
        const int hi = (int)fminf(fmaxf(rintf(__fdiv_rn(V[1][r], vsc[r])), -8.f), 7.f);
        vrow[r * (PK_D / 2) + lane] = (uint8_t)((lo & 15) | ((hi & 15) << 4));
        if (lane == r) reinterpret_cast<uint16_t*>(S.vs + row * S.svs)[r] = f32_to_bf16(vsc[r]);
    }
    // coefficients: lane t < PK_PG owns token t
    if (lane < PK_PG) {
        const int t = lane;
        float C[BD_RNK];
        float am = 0.f;
#pragma unroll
        for (int r = 0; r < BD_RNK; ++r) {
            C[r] = __fmul_rn(L.U[t][PK_PG - BD_RNK + r], L.S8[r]);
            am = fmaxf(am, fabsf(C[r]));
        }
        const float csc = fmaxf(__fdiv_rn(am, 127.f), 1e-8f);
        int8_t* crow = reinterpret_cast<int8_t*>(S.c8 + row * S.sc8) + t * BD_RNK;
#pragma unroll
        for (int r = 0; r < BD_RNK; ++r)
            crow[r] = (int8_t)fminf(fmaxf(rintf(__fdiv_rn(C[r], csc)), -127.f), 127.f);
        reinterpret_cast<uint16_t*>(S.cs + row * S.scs)[t] = f32_to_bf16(csc);
    }
    // centroid
    const float msc = fmaxf(__fdiv_rn(wave_max(fmaxf(fabsf(L.mu[2 * lane]), fabsf(L.mu[2 * lane + 1]))), 127.f), 1e-8f);
#pragma unroll
    for (int e = 0; e < 2; ++e)
        reinterpret_cast<int8_t*>(S.mu + row * S.smu)[2 * lane + e] =
            (int8_t)fminf(fmaxf(rintf(__fdiv_rn(L.mu[2 * lane + e], msc)), -127.f), 127.f);
    if (lane == 0) *reinterpret_cast<uint16_t*>(S.mus + row * S.smus) = f32_to_bf16(msc);
}

__global__ __launch_bounds__(4 * kWave) void rki4_pack_kernel(
    const float* __restrict__ mu, const float* __restrict__ dc, const float* __restrict__ S2,
    const float* __restrict__ U, const int* __restrict__ rows, int n, SlabRows S)
{
    __shared__ PackLds lds[4];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    PackLds& L = lds[wave];
    const long item = (long)blockIdx.x * 4 + wave;
    if (item >= n) return;
    for (int i = lane; i < PK_PG * PK_D; i += kWave) L.dc[i / PK_D][i % PK_D] = dc[item * PK_PG * PK_D + i];
    for (int i = lane; i < PK_D; i += kWave) L.mu[i] = mu[item * PK_D + i];
    for (int i = lane; i < PK_PG * PK_PG; i += kWave) L.U[i / PK_PG][i % PK_PG] = U[item * PK_PG * PK_PG + i];
    if (lane < BD_RNK) L.S8[lane] = __fsqrt_rn(fmaxf(S2[item * PK_PG + PK_PG - BD_RNK + lane], 1e-10f));
    wave_lds_sync();
    pack_page(L, rows[item], S);
}

// ---- refresh lifecycle: which blocks to (re)build --------------------------
// Reference producers: selection/build.py:372-384 _tail_blocks, :415-427
// _bulk_blocks, :472-488 _delta_select (rki4_build.py:264-315 call them).
// One thread per candidate page marks its physical block in a byte map
// (duplicates collapse: pages shared by several requests are built once);
// refresh_compact_kernel turns the map into a list plus a device count and
// clears the map again.  No host sync on any mode.
constexpr int RF_THREADS = 256;

__device__ __forceinline__ bool tags_differ(uint4 a, uint4 b) {
    // bf16 values compared as numbers, like the reference's float compare:
    // NaN (the never-built tag) differs from everything, -0 equals +0
    const uint32_t wa[4] = {a.x, a.y, a.z, a.w}, wb[4] = {b.x, b.y, b.z, b.w};
    bool d = false;
#pragma unroll
    for (int e = 0; e < 4; ++e)
        d |= (bf16lo(wa[e]) != bf16lo(wb[e])) | (bf16hi(wa[e]) != bf16hi(wb[e]));
    return d;
}

__global__ __launch_bounds__(RF_THREADS) void refresh_mark_kernel(
    int mode, const int* __restrict__ bt, long bt_sr, const int* __restrict__ sl, int n_req,
    const int* __restrict__ rows, int n_rows, int max_fin, int page, int NB,
    const uint64_t* __restrict__ k_layers, long k_sb, long k_st, long k_sh, int n_kv,
    const uint16_t* __restrict__ tag, long layer_rows, uint8_t* __restrict__ mark,
    int* __restrict__ count)
{
    const long i = (long)blockIdx.x * RF_THREADS + threadIdx.x;
    if (i == 0 && blockIdx.y == 0) *count = 0;           // compact runs after this kernel
    // delta: one thread per (page, kv head), heads of one page adjacent
    const int kh = mode == LOCKS_REFRESH_DELTA ? (int)(i % n_kv) : 0;
    const long pi = mode == LOCKS_REFRESH_DELTA ? i / n_kv : i;
    int blk;
    if (mode == LOCKS_REFRESH_TAIL) {
        if (pi >= n_rows) return;
        const int r = rows ? rows[pi] : (int)pi;
        if (r < 0 || r >= n_req) return;
        const int fin1 = min(max(sl[r] / page - 1, 0), (int)bt_sr - 1);   // last finalized page
        blk = bt[(long)r * bt_sr + fin1];
    } else {
        if (pi >= (long)n_req * max_fin) return;
        const int r = (int)(pi / max_fin), p = (int)(pi % max_fin);
        if (p >= sl[r] / page) return;                    // not finalized
        blk = bt[(long)r * bt_sr + p];
    }
    if (blk < 0 || blk >= NB) return;
    if (mode == LOCKS_REFRESH_DELTA) {
        const int layer = blockIdx.y;
        const uint16_t* kp = reinterpret_cast<const uint16_t*>(k_layers[layer]) +
                             (long)blk * k_sb + (long)(page - 1) * k_st + (long)kh * k_sh;
        const uint16_t* tp = tag + ((long)layer * layer_rows + (long)blk * n_kv + kh) * 8;
        if (!tags_differ(*reinterpret_cast<const uint4*>(kp), *reinterpret_cast<const uint4*>(tp)))
            return;
    }
    mark[blk] = 1;
}

__global__ __launch_bounds__(RF_THREADS) void refresh_compact_kernel(
    uint8_t* __restrict__ mark, int NB, int* __restrict__ blocks, int* __restrict__ count)
{
    const int i = blockIdx.x * RF_THREADS + threadIdx.x;
    const int lane = threadIdx.x & 63;
    const bool m = i < NB && mark[i] != 0;
    if (m) mark[i] = 0;
    const uint64_t bal = __ballot(m);
    if (bal == 0) return;
    const int pre = __builtin_amdgcn_mbcnt_hi((uint32_t)(bal >> 32),
                                              __builtin_amdgcn_mbcnt_lo((uint32_t)bal, 0u));
    int base = 0;
    if (lane == 0) base = atomicAdd(count, __popcll(bal));
    base = __shfl(base, 0);
    if (m) blocks[base + pre] = i;
}

// Tail mode for up to RF_THREADS rows in one launch: one workgroup takes each
// row's last finalized page and lists each block once.  The byte map is not
// needed (marking and compacting it took two launches for a handful of rows:
// tail of 4 requests, 32 layers, 59.9 -> 56.9 us).  Duplicates collapse in an
// LDS hash table, whose time does not grow with the rows: two launches 3.7 / 4.4 /
// 6.5 us at 4 / 64 / 256 rows, this one 2.1 / 2.1 / 2.3 (with each row compared to
// all earlier ones 2.2 / 5.2 / 14.8).  Two multiplications spread blocks at any
// regular distance (a table's width): 256 of them probe 17 slots at worst for
// distances up to 4200 (one multiplication: 256).  There are at most RF_THREADS
// blocks in RF_SLOTS slots, so a probe ends at its block or at a free slot.
constexpr int RF_SLOT_BITS = 10, RF_SLOTS = 1 << RF_SLOT_BITS;
static_assert(RF_SLOTS == 4 * RF_THREADS, "four slots a thread");
__global__ __launch_bounds__(RF_THREADS) void refresh_tail_kernel(
    const int* __restrict__ bt, long bt_sr, const int* __restrict__ sl, int n_req,
    const int* __restrict__ rows, int n_rows, int page, int NB, int* __restrict__ blocks,
    int* __restrict__ count)
{
    __shared__ __attribute__((aligned(16))) int slot[RF_SLOTS];
    __shared__ int n;
    const int i = threadIdx.x;
    int blk = -1;
    if (i < n_rows) {
        const int r = rows ? rows[i] : i;
        if (r >= 0 && r < n_req) {
            const int fin1 = min(max(sl[r] / page - 1, 0), (int)bt_sr - 1);   // last finalized page
            blk = bt[(long)r * bt_sr + fin1];
        }
    }
    *reinterpret_cast<int4*>(&slot[4 * i]) = make_int4(-1, -1, -1, -1);
    if (i == 0) n = 0;
    __syncthreads();
    if (blk >= 0 && blk < NB) {
        uint32_t h = (uint32_t)blk * 0x9E3779B1u;
        h = (h ^ (h >> 15)) * 0x85EBCA77u;
        for (int at = (int)(h >> (32 - RF_SLOT_BITS));; at = (at + 1) & (RF_SLOTS - 1)) {
            const int had = atomicCAS(&slot[at], -1, blk);
            if (had == -1) blocks[atomicAdd(&n, 1)] = blk;           // this row is the first with the block
            if (had == -1 || had == blk) break;
        }
    }
    __syncthreads();
    if (i == 0) *count = n;
}

}  // namespace locks

using namespace locks;

// (head_dim, page) of the summary builder: {64, 128, 256} x {16, 32, 64}
// (the reference's rki4 geometry domain, rki4_state.py:295-324) plus the MLA
// latent (512, 16).
static bool bd_geometry(int head_dim, int page) {
    if (head_dim == 512) return page == 16;
    return (head_dim == 64 || head_dim == 128 || head_dim == 256) && (page == 16 || page == 32 || page == 64);
}
template <int D, int PG>
static int bd_launch(const uint16_t* kc, const uint64_t* k_layers, long k_sb, long k_st, long k_sh,
                     int NB, const int* blocks, const int* count, int n_blocks, int n_kv,
                     int n_layers, long layer_rows, const SlabRows& S, uint16_t* tag, hipStream_t st) {
    const long items = (long)n_blocks * n_kv * n_layers;
    const int gpw = pages_per_wave(items, BD_SPREAD, kWave / PG);
    const long grid = std::min((items + 4 * gpw - 1) / (4 * gpw), BD_MAX_GRID);
    hipLaunchKernelGGL((rki4_build_kernel<D, PG>), dim3((unsigned)grid), dim3(4 * kWave), 0, st, kc,
                       k_layers, k_sb, k_st, k_sh, NB, blocks, count, n_blocks, n_kv, n_layers,
                       layer_rows, S, tag);
    return check_launch("rki4_build_kernel");
}
#define BD_DISPATCH(HD, PGV, ...)                                              \
    ((HD) == 512 ? bd_launch<512, 16>(__VA_ARGS__)                               \
     : (PGV) == 16 ? ((HD) == 128 ? bd_launch<128, 16>(__VA_ARGS__)              \
                      : (HD) == 64 ? bd_launch<64, 16>(__VA_ARGS__)              \
                                   : bd_launch<256, 16>(__VA_ARGS__))            \
     : (PGV) == 32 ? ((HD) == 128 ? bd_launch<128, 32>(__VA_ARGS__)              \
                      : (HD) == 64 ? bd_launch<64, 32>(__VA_ARGS__)              \
                                   : bd_launch<256, 32>(__VA_ARGS__))            \
                   : ((HD) == 128 ? bd_launch<128, 64>(__VA_ARGS__)              \
                      : (HD) == 64 ? bd_launch<64, 64>(__VA_ARGS__)              \
                                   : bd_launch<256, 64>(__VA_ARGS__)))

extern "C" int32_t locks_build_rki4(
    const uint16_t* k_cache, int64_t k_stride_block, int64_t k_stride_tok, int64_t k_stride_head,
    int32_t num_blocks, const int32_t* blocks, int32_t n_blocks, int32_t n_kv, int32_t head_dim,
    int32_t page, uint8_t* v4, uint16_t* vs, int8_t* c8, uint16_t* cs, int8_t* mu8,
    uint16_t* mus, const int64_t* slab_row_bytes, uint16_t* tag, void* stream)
{
    LOCKS_REQUIRE(bd_geometry(head_dim, page),
                  "locks_build_rki4: geometry d=%d page=%d unsupported (d 64/128/256 with page 16/32/64, "
                  "or d 512 with page 16)", head_dim, page);
    LOCKS_REQUIRE(n_kv >= 1 && num_blocks >= 1 && n_blocks >= 0, "locks_build_rki4: bad geometry");
    LOCKS_REQUIRE(k_stride_tok % 8 == 0 && k_stride_block % 8 == 0 && k_stride_head % 8 == 0,
                  "locks_build_rki4: K strides must be multiples of 8 elements");
    LOCKS_REQUIRE(k_cache && blocks && v4 && vs && c8 && cs && mu8 && mus && tag,
                  "locks_build_rki4: null pointer argument");
    const SlabRows S = slab_rows(v4, vs, c8, cs, mu8, mus, slab_row_bytes, head_dim, page);
    LOCKS_REQUIRE(slab_rows_ok(S, head_dim, page),
                  "locks_build_rki4: slab row strides below the field sizes or misaligned");
    if (n_blocks == 0) return 0;
    return BD_DISPATCH(head_dim, page, k_cache, nullptr, (long)k_stride_block, (long)k_stride_tok,
                       (long)k_stride_head, num_blocks, blocks, nullptr, n_blocks, n_kv, 1, 0L,
                       S, tag, (hipStream_t)stream);
}

extern "C" int32_t locks_pack_rki4(const float* mu, const float* dc, const float* S2,
                                   const float* U, const int32_t* rows, int32_t n,
                                   int32_t head_dim, int32_t page, uint8_t* v4, uint16_t* vs,
                                   int8_t* c8, uint16_t* cs, int8_t* mu8, uint16_t* mus,
                                   const int64_t* slab_row_bytes, void* stream)
{
    LOCKS_REQUIRE(head_dim == PK_D && page == PK_PG,
                  "locks_pack_rki4: geometry d=%d page=%d unsupported (this entry: 128/16)", head_dim, page);
    LOCKS_REQUIRE(n >= 0, "locks_pack_rki4: n=%d < 0", n);
    LOCKS_REQUIRE(mu && dc && S2 && U && rows && v4 && vs && c8 && cs && mu8 && mus,
                  "locks_pack_rki4: null pointer argument");
    const SlabRows S = slab_rows(v4, vs, c8, cs, mu8, mus, slab_row_bytes, head_dim, page);
    LOCKS_REQUIRE(slab_rows_ok(S, head_dim, page),
                  "locks_pack_rki4: slab row strides below the field sizes or misaligned");
    if (n == 0) return 0;
    hipLaunchKernelGGL(rki4_pack_kernel, dim3((n + 3) / 4), dim3(4 * kWave),
                       0, (hipStream_t)stream, mu, dc, S2, U, rows, n, S);
    return check_launch("rki4_pack_kernel");
}

extern "C" int32_t locks_refresh_blocks(
    int32_t mode, const int32_t* block_table, int64_t bt_stride, const int32_t* seq_lens,
    int32_t n_req, const int32_t* rows, int32_t n_rows, int32_t max_fin, int32_t page,
    int32_t num_blocks, const uint64_t* k_layers, int32_t n_layers, int64_t k_stride_block,
    int64_t k_stride_tok, int64_t k_stride_head, int32_t n_kv, const uint16_t* tag,
    int64_t tag_blocks, uint8_t* mark, int32_t* blocks, int32_t* count, void* stream)
{
    LOCKS_REQUIRE(mode == LOCKS_REFRESH_TAIL || mode == LOCKS_REFRESH_BULK ||
                      mode == LOCKS_REFRESH_DELTA,
                  "locks_refresh_blocks: unknown mode %d", mode);
    LOCKS_REQUIRE(block_table && seq_lens && mark && blocks && count,
                  "locks_refresh_blocks: null pointer argument");
    LOCKS_REQUIRE(n_req >= 0 && n_rows >= 0 && max_fin >= 0 && page >= 1 && num_blocks >= 1 &&
                      bt_stride >= 1,
                  "locks_refresh_blocks: bad geometry");
    if (mode == LOCKS_REFRESH_BULK || mode == LOCKS_REFRESH_DELTA)
        LOCKS_REQUIRE(max_fin <= bt_stride, "locks_refresh_blocks: max_fin %d > block-table width %lld",
                      max_fin, (long long)bt_stride);
    if (mode == LOCKS_REFRESH_DELTA) {
        LOCKS_REQUIRE(k_layers && tag && n_layers >= 1 && n_layers <= 65535 && n_kv >= 1 &&
                          tag_blocks >= num_blocks,
                      "locks_refresh_blocks: delta needs k_layers, tag, n_layers, n_kv");
        LOCKS_REQUIRE(k_stride_tok % 8 == 0 && k_stride_block % 8 == 0 && k_stride_head % 8 == 0,
                      "locks_refresh_blocks: K strides must be multiples of 8 elements");
    }
    if (mode == LOCKS_REFRESH_TAIL && n_rows <= RF_THREADS) {
        hipLaunchKernelGGL(refresh_tail_kernel, dim3(1), dim3(RF_THREADS), 0, (hipStream_t)stream, block_table,
                           (long)bt_stride, seq_lens, n_req, rows, n_rows, page, num_blocks, blocks, count);
        return check_launch("refresh_tail_kernel");
    }
    const long items = mode == LOCKS_REFRESH_TAIL ? (long)n_rows
                       : (long)n_req * max_fin * (mode == LOCKS_REFRESH_DELTA ? n_kv : 1);
    const long gx = std::max<long>(1, (items + RF_THREADS - 1) / RF_THREADS);
    LOCKS_REQUIRE(gx < (1L << 31), "locks_refresh_blocks: too many pages in one call");
    const int gy = mode == LOCKS_REFRESH_DELTA ? n_layers : 1;
    hipLaunchKernelGGL(refresh_mark_kernel, dim3((unsigned)gx, gy), dim3(RF_THREADS), 0,
                       (hipStream_t)stream, mode, block_table, (long)bt_stride, seq_lens, n_req,
                       rows, n_rows, max_fin, page, num_blocks, k_layers, (long)k_stride_block,
                       (long)k_stride_tok, (long)k_stride_head, n_kv, tag,
                       (long)tag_blocks * n_kv, mark, count);
    int32_t rc = check_launch("refresh_mark_kernel");
    if (rc) return rc;
    hipLaunchKernelGGL(refresh_compact_kernel, dim3((num_blocks + RF_THREADS - 1) / RF_THREADS),
                       dim3(RF_THREADS), 0, (hipStream_t)stream, mark, num_blocks, blocks, count);
    return check_launch("refresh_compact_kernel");
}

extern "C" int32_t locks_build_rki4_layers(
    const uint64_t* k_layers, int32_t n_layers, int64_t k_stride_block, int64_t k_stride_tok,
    int64_t k_stride_head, int32_t num_blocks, const int32_t* blocks, const int32_t* count,
    int32_t n_blocks, int32_t n_kv, int32_t head_dim, int32_t page, int64_t slab_blocks,
    uint8_t* v4, uint16_t* vs, int8_t* c8, uint16_t* cs, int8_t* mu8, uint16_t* mus,
    const int64_t* slab_row_bytes, uint16_t* tag, void* stream)
{
    LOCKS_REQUIRE(bd_geometry(head_dim, page),
                  "locks_build_rki4_layers: geometry d=%d page=%d unsupported (d 64/128/256 with page "
                  "16/32/64, or d 512 with page 16)", head_dim, page);
    LOCKS_REQUIRE(n_kv >= 1 && num_blocks >= 1 && n_blocks >= 0 && n_layers >= 1 &&
                      n_layers <= 65535 && slab_blocks >= num_blocks,
                  "locks_build_rki4_layers: bad geometry");
    LOCKS_REQUIRE(k_stride_tok % 8 == 0 && k_stride_block % 8 == 0 && k_stride_head % 8 == 0,
                  "locks_build_rki4_layers: K strides must be multiples of 8 elements");
    LOCKS_REQUIRE(k_layers && blocks && v4 && vs && c8 && cs && mu8 && mus && tag,
                  "locks_build_rki4_layers: null pointer argument");
    const SlabRows S = slab_rows(v4, vs, c8, cs, mu8, mus, slab_row_bytes, head_dim, page);
    LOCKS_REQUIRE(slab_rows_ok(S, head_dim, page),
                  "locks_build_rki4_layers: slab row strides below the field sizes or misaligned");
    if (n_blocks == 0) return 0;
    const long layer_rows = (long)slab_blocks * n_kv;
    return BD_DISPATCH(head_dim, page, nullptr, k_layers, (long)k_stride_block, (long)k_stride_tok,
                       (long)k_stride_head, num_blocks, blocks, count, n_blocks, n_kv, n_layers,
                       layer_rows, S, tag, (hipStream_t)stream);
}
