// gam_net.hip -- the learned coarse-grid correction: a 3-layer 3x3x3 conv net
// (8 -> 32 -> 32 -> 8 channels, leaky ReLU between) on the ghost-inclusive cell grid,
// with BF16 weights and activations and FP32 accumulation on gfx950's
// v_mfma_f32_16x16x32_bf16.  Forward, backward (data and weights) and Adam are
// hand-written here; libgamera_net.so exports them (include/gamera_net.h).
//
// Layouts (nc = cells of the ghost-inclusive box, p = linear cell index, i fastest):
//   activations  act[p][32]   BF16, channels last
//   weights      W[l][tap][co][ci] BF16 (ci = 32 padded), tap = dz*9 + dy*3 + dx;
//                the first layer (8 input channels) packs 4 taps per K = 32:
//                W0[g][co][4*8] with taps 4g..4g+3 (zero past tap 26)
//   output       out[p][8]    FP32 (the correction field, channels last)
// A convolution is an implicit GEMM: M = 16 consecutive cells per MFMA, N = 16
// output channels per tile, K = 32 input channels of one tap per MFMA (of four
// taps in the first layer).  Output
// cells cover [lo, nc - lo) with lo = Ni*Nj + Ni + 1, the cells whose every tap's
// neighbour p + off lies inside the array; cells near the box faces read
// wrapped neighbours and are never used (the correction is read on the active
// box plus one layer only, 4 ghost layers deep).
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <algorithm>
#include <string>
#include <type_traits>
#include <vector>
#include <cstring>
#include <cmath>

#include "gamera_net.h"

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef unsigned short u16;

#define NET_C 32      // padded channel count of every activation
#define NET_TAPS 27
#define NET_G0 7      // K steps of the first layer: ceil(27 taps / 4)
#define NET_LEAK 0.125f

// round-to-nearest-even FP32 -> BF16 (finite inputs)
__host__ __device__ inline u16 f2bf(float f) {
    uint32_t u;
    memcpy(&u, &f, 4);
    uint32_t r = u + 0x7FFFu + ((u >> 16) & 1u);
    return (u16)(r >> 16);
}
__host__ __device__ inline float bf2f(u16 b) {
    uint32_t u = (uint32_t)b << 16;
    float f;
    memcpy(&f, &u, 4);
    return f;
}

struct NetDims { int Ni, Nj, Nk, nc, lo, hi; };   // computed cells [lo, hi)

__device__ __forceinline__ bf16x8 ld8(const u16 *p) {   // 16-byte aligned
    return *reinterpret_cast<const bf16x8 *>(p);
}

// ----------------------------------------------------------------- convolution
// The training convolutions (k_conv) and the inference (k_infer below) work on bricks of
// NB_I x NB_J x NB_K cells, tiles of 16 cells along i.  A brick's input, the brick and
// one cell around it, is staged once in LDS (80 bytes per cell of 32 channels: the
// lanes of a 16-byte read fall on distinct banks), so an input cell comes from L2 2.5
// times instead of once per tap.
// CIN = 8: a wave has the tiles of one k row and all output channels, and packs 4 taps
// per K step (lane group kg reading tap 4s + kg).
// CIN = 32, one tap per K step: a wave has one 16-channel output tile on NCO / 16 k rows, so
// its weights of all 27 taps fit its registers (108), and blocks stay
// for several bricks, the next one's input on its way to registers meanwhile.  Fetched per
// brick, the 55 KB of weights passed the 32 KB L1 for every 64 cells, and the MFMAs
// waited for them.  The tile rows of a staged plane are each read once for
// the up to 3 x NCO / 16 output rows that they feed.
// The taps add in the order dx, dy, dz in either form.
#define NB_I 16
#define NB_J 4
#define NB_K 4
#define NB_LI (NB_I + 2)
#define NB_LJ (NB_J + 2)
#define NB_LK (NB_K + 2)
#define NB_LC (NB_LI * NB_LJ * NB_LK)   // staged cells
#define NB_OC (NB_I * NB_J * NB_K)      // output cells
#define NB_STAY 512   // blocks of the 32-channel kernels: 2 on each of 256 CUs

template <int CIN, int NCO>
struct ConvT {
    static constexpr int CS = CIN == 32 ? 40 : 8;           // BF16 elements per staged cell
    static constexpr int OS = 40;                           // and per output cell of 32 channels: 80 bytes
    static constexpr int TW = CIN == 32 ? 1 : NCO / 16;     // output tiles per wave
    static constexpr int KT = CIN == 32 ? NCO / 16 : 1;     // k rows per wave
    static constexpr int NS = CIN == 32 ? NET_TAPS : (NET_TAPS + 3) / 4;   // K steps
    bf16x8 w[CIN == 32 ? NS : 2][TW];   // CIN = 8: two K steps ahead
    f32x4 acc[KT][NB_J][TW];
    const u16 *W;
    int row, kg, t0, kr;   // lane's row and K group; the wave's first output tile and k row
    __device__ __forceinline__ bf16x8 weight(int q, int t) const {
        return ld8(W + (size_t)(q * NCO + 16 * (t0 + t) + row) * NET_C + 8 * kg);
    }
    __device__ __forceinline__ void init(const u16 *W_) {
        const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
        W = W_;
        row = lane & 15; kg = lane >> 4;
        t0 = CIN == 32 ? wave % (NCO / 16) : 0;
        kr = CIN == 32 ? wave / (NCO / 16) * KT : wave;
#pragma unroll
        for (int q = 0; q < (CIN == 32 ? NS : 2); q++)
#pragma unroll
            for (int t = 0; t < TW; t++) w[q][t] = weight(q, t);
    }
    __device__ __forceinline__ void run(const u16 *sA) {
#pragma unroll
        for (int q = 0; q < KT * NB_J * TW; q++) acc[q / (NB_J * TW)][(q / TW) % NB_J][q % TW] = f32x4{0.f, 0.f, 0.f, 0.f};
        if constexpr (CIN == 8) {
#pragma unroll 1
            for (int st = 0; st < NS; st++) {
                const int tap = 4 * st + kg;
                const bool live = tap < NET_TAPS;   // K slots past the last tap: zero A (their weights are zero too)
                const int tp = live ? tap : 13;     // a staged cell for the dead slots
                const int c0 = (kr + tp / 9) * (NB_LJ * NB_LI) + ((tp / 3) % 3) * NB_LI + tp % 3 + row;
                bf16x8 bw[TW];
                const int sn = st + 2 < NS ? st + 2 : NS - 1;
#pragma unroll
                for (int t = 0; t < TW; t++) { bw[t] = w[0][t]; w[0][t] = w[1][t]; w[1][t] = weight(sn, t); }
#pragma unroll
                for (int m = 0; m < NB_J; m++) {
                    bf16x8 a = *reinterpret_cast<const bf16x8 *>(sA + (size_t)(c0 + m * NB_LI) * CS);
                    if (!live) a = bf16x8{};
#pragma unroll
                    for (int t = 0; t < TW; t++) acc[0][m][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, bw[t], acc[0][m][t], 0, 0, 0);
                }
            }
        } else {
            // the staged tile rows (plane pl, row r) in turn, each read one row ahead; row r of
            // plane pl is the tap (dy, dz) = (r - m, pl - kt) - 1 of output row m, k row kt
            const u16 *s0 = sA + (size_t)(kr * (NB_LJ * NB_LI) + row) * CS + 8 * kg;
            bf16x8 a[2][3];
            auto rd = [&](int n) {
#pragma unroll
                for (int dx = 0; dx < 3; dx++) a[n & 1][dx] = *reinterpret_cast<const bf16x8 *>(s0 + (n * NB_LI + dx) * CS);
            };
            rd(0);
#pragma unroll
            for (int n = 0; n < (KT + 2) * NB_LJ; n++) {
                if (n + 1 < (KT + 2) * NB_LJ) rd(n + 1);
                const int pl = n / NB_LJ, r = n % NB_LJ;
#pragma unroll
                for (int kt = 0; kt < KT; kt++)
#pragma unroll
                    for (int m = 0; m < NB_J; m++) {
                        if (pl - kt < 0 || pl - kt > 2 || r - m < 0 || r - m > 2) continue;
#pragma unroll
                        for (int dx = 0; dx < 3; dx++)
                            acc[kt][m][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[n & 1][dx], w[9 * (pl - kt) + 3 * (r - m) + dx][0],
                                                                                    acc[kt][m][0], 0, 0, 0);
                    }
                __builtin_amdgcn_sched_barrier(0);   // no reads hoisted further: registers
            }
        }
    }
};

// Bricks of a block: the launch's bricks in 8 runs, one per XCD, whose L2 then holds
// the neighbours' shared cells.
__device__ __forceinline__ int brick_run(int nbrick) { return (nbrick + 7) / 8; }
static unsigned brick_blocks(long nbrick, long most) { return (unsigned)std::min((nbrick + 7) / 8 * 8, most); }

// 8 BF16 gradients times the slope at the forward outputs m (1/8: exact, so before or after the rounding)
__device__ __forceinline__ uint4 masked(const uint4 &x, const uint4 &m) {
    const uint32_t xw[4] = {x.x, x.y, x.z, x.w}, mw[4] = {m.x, m.y, m.z, m.w};
    uint32_t o[4];
#pragma unroll
    for (int h = 0; h < 4; h++) {
        float l = bf2f((u16)(xw[h] & 0xFFFFu)), u = bf2f((u16)(xw[h] >> 16));
        if (bf2f((u16)(mw[h] & 0xFFFFu)) <= 0.f) l = NET_LEAK * l;
        if (bf2f((u16)(mw[h] >> 16)) <= 0.f) u = NET_LEAK * u;
        o[h] = (uint32_t)f2bf(l) | ((uint32_t)f2bf(u) << 16);
    }
    return uint4{o[0], o[1], o[2], o[3]};
}

// Hidden activation: leaky ReLU, x > 0 ? x : x/8 (a slope that keeps every
// unit trainable; 1/8 is exact in BF16 and FP32).
// MODE 0: activation, write act_out, NCO = 32
// MODE 1: linear output, write out[p][0..7] FP32 (NCO = 16, channels 8..15 padding)
// MODE 2: backward data: multiply by the activation's slope at the forward
//         output (mask > 0: 1, else 1/8), write act_out, NCO = 32
// Neighbours are those of the flattened cell index (p + off), as at the box faces, whose
// cells are never used; cells outside [lo, hi) are not stored.  The results leave
// through LDS as whole cells.
// Per launch on a 104^3 grid, A operands from L2 / staged, weights per brick / as now:
// hidden layer 230 / 151 / 69 us, first 111 / 84 / 49, last 182 / 70 / 43, backward
// data 272 / 192 / 79.  Of that the channel-major copies that the weight gradients once
// read were 25, 13, 0 and 52.
template <int CIN, int NCO, int MODE>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(CIN == 32 ? 2 : 4)))
k_conv(NetDims d, const u16 *__restrict__ in, const u16 *__restrict__ W, const float *__restrict__ bias,
       const u16 *__restrict__ mask, u16 *__restrict__ act_out, float *__restrict__ out) {
    static_assert(CIN == 8 || CIN == 32, "8 or 32 input channels");
    static_assert(NB_I == 16 && NB_K == 4, "one 16-cell tile per row, four waves on four k rows");
    using T = ConvT<CIN, NCO>;
    constexpr int CS = T::CS, OS = T::OS, PER = CIN / 8;   // PER: 16-byte pieces per cell
    constexpr int NIT = (NB_LC * PER + 255) / 256;
    __shared__ uint4 sIn[NB_LC * CS / 8];
    __shared__ uint4 sOut[MODE == 1 ? NB_OC * 2 : NB_OC * OS / 8];
    u16 *sO = reinterpret_cast<u16 *>(sOut);
    float *sF = reinterpret_cast<float *>(sOut);
    const int nbi = (d.Ni + NB_I - 1) / NB_I, nbj = (d.Nj + NB_J - 1) / NB_J, nbk = (d.Nk + NB_K - 1) / NB_K;
    const int run = brick_run(nbi * nbj * nbk);
    const int b0 = (blockIdx.x & 7) * run, b1 = min(b0 + run, nbi * nbj * nbk), step = gridDim.x >> 3;
    int b = b0 + (blockIdx.x >> 3);
    auto origin = [&](int bb, int &oi, int &oj, int &ok) { oi = NB_I * (bb % nbi); oj = NB_J * ((bb / nbi) % nbj); ok = NB_K * (bb / (nbi * nbj)); };
    uint4 v[NIT];
    auto fetch = [&](int bb) {
        int oi, oj, ok;
        origin(bb, oi, oj, ok);
#pragma unroll
        for (int it = 0; it < NIT; it++) {
            const int e = threadIdx.x + 256 * it, c = e / PER;
            const int li = c % NB_LI, lj = (c / NB_LI) % NB_LJ, lk = c / (NB_LI * NB_LJ);
            const int p = (oi - 1 + li) + d.Ni * ((oj - 1 + lj) + d.Nj * (ok - 1 + lk));
            v[it] = uint4{0u, 0u, 0u, 0u};
            if (c < NB_LC && p >= 0 && p < d.nc) v[it] = *reinterpret_cast<const uint4 *>(in + (size_t)p * NET_C + 8 * (e % PER));
        }
    };
    if (b >= b1) return;
    fetch(b);
    T cv;
    cv.init(W);
    for (; b < b1; b += step) {
#pragma unroll
        for (int it = 0; it < NIT; it++) {
            const int e = threadIdx.x + 256 * it, c = e / PER;
            if (c < NB_LC) sIn[c * (CS / 8) + e % PER] = v[it];
        }
        __syncthreads();   // staged; and every wave has read the last brick's sOut
        if (CIN == 32 && b + step < b1) fetch(b + step);
        cv.run(reinterpret_cast<const u16 *>(sIn));
        int oi, oj, ok;
        origin(b, oi, oj, ok);
#pragma unroll
        for (int q = 0; q < T::KT * NB_J * T::TW; q++) {
            const int kt = q / (NB_J * T::TW), m = (q / T::TW) % NB_J, t = q % T::TW;
            const int co = 16 * (cv.t0 + t) + cv.row, kk = cv.kr + kt, oc = (kk * NB_J + m) * NB_I + 4 * cv.kg;
            const f32x4 x = cv.acc[kt][m][t];
            if constexpr (MODE == 1) {
                if (co < 8) {
                    const float bb = bias[co];
#pragma unroll
                    for (int r = 0; r < 4; r++) sF[(oc + r) * 8 + co] = x[r] + bb;
                }
            } else {
                const float bb = MODE == 0 ? bias[co] : 0.f;
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    float y = x[r];
                    if constexpr (MODE == 0) { y += bb; y = y > 0.f ? y : NET_LEAK * y; }
                    sO[(oc + r) * OS + co] = f2bf(y);
                }
            }
        }
        __syncthreads();   // results in sOut; and every wave is done with sIn
        constexpr int CH = MODE == 1 ? 2 : 4;   // 16-byte pieces per output cell
        for (int e = threadIdx.x; e < NB_OC * CH; e += 256) {
            const int oc = e / CH, q = e % CH;
            const int i = oi + oc % NB_I, j = oj + (oc / NB_I) % NB_J, k = ok + oc / (NB_I * NB_J), p = i + d.Ni * (j + d.Nj * k);
            if (i >= d.Ni || j >= d.Nj || k >= d.Nk || p < d.lo || p >= d.hi) continue;
            if constexpr (MODE == 1) *reinterpret_cast<uint4 *>(out + (size_t)p * 8 + 4 * q) = sOut[e];
            else {
                uint4 x = sOut[oc * (OS / 8) + q];
                if constexpr (MODE == 2) x = masked(x, *reinterpret_cast<const uint4 *>(mask + (size_t)p * NET_C + 8 * q));
                *reinterpret_cast<uint4 *>(act_out + (size_t)p * NET_C + 8 * q) = x;
            }
        }
    }
}

// Weight and bias gradients of one layer, dW[tap][co][ci] += sum_p g[p][co] *
// a[p + off][ci] and db[co] += sum_p g[p][co]: per tap a GEMM with M = output
// channels, N = input channels and K = cells.  Both operands are staged channels
// last, a brick of gradients and the activations one cell around it, and read with
// the transposing LDS read (ds_read_b64_tr_b16: lane l of 16 gets column l of 4 rows of
// 16): a row of 16 cells is half of a K step of any dx, a step is the rows j, j + 2, and a pair
// of activation rows serves up to two steps and three k rows.  So a brick is
// read from memory 2.5 times, not 9, and needs no channel-major copy of either array.
// A wave keeps the 27 taps of one 16 x 16 tile (108 accumulator registers) on
// KK of the brick's 4 k rows; the bias is one more MFMA against ones.  The two LDS buffers
// alternate: the next brick's loads are in flight while this one's MFMAs run.
// Per wave and brick (MT = NT = 2) 108 MFMAs on 112 8-byte reads: the LDS and the
// matrix units are about equally busy.  The block's waves add up in LDS, and the
// block writes its sums to a workspace that k_wreduce adds in a fixed order, so the
// gradients do not depend on the order blocks finish in.  Cells outside the
// computed range carry a zero gradient (never written, zero from allocation).
// Per launch on a 104^3 grid, layers 2 / 1 / 0: 463 / 813 / 435 us with one tap per wave,
// 187 / 231 / 119 with channel-major rows from L2 -> 55 / 77 / 52, and 5 for the sums (18 before).
#define WG_BLOCKS 256   // one per CU: 2 waves per SIMD
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef bf16x4 __attribute__((address_space(3))) lds_bf16x4;
__device__ __forceinline__ bf16x8 tr_rows(const u16 *a, const u16 *b) {   // 4 + 4 cells of a channel
    const bf16x4 x = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4 *)a), y = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4 *)b);
    return __builtin_shufflevector(x, y, 0, 1, 2, 3, 4, 5, 6, 7);
}

template <int MT, int NT>
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2)))
k_wgrad(NetDims d, const u16 *__restrict__ g, const u16 *__restrict__ act, float *__restrict__ ws) {
    static_assert(NB_I == 16 && NB_J == 4 && NB_K == 4, "two K steps of two rows per k row");
    constexpr int PA = 2 * NT, PG = 2 * MT;                   // 16-byte pieces per staged cell
    constexpr int SA = NT == 2 ? 40 : 24, SG = MT == 2 ? 40 : 24;   // BF16 elements per staged cell: rows fall on distinct banks
    constexpr int NA = NB_LC * PA, NG = NB_OC * PG, NIT = (NA + NG + 511) / 512;
    constexpr int KS = 8 / (MT * NT), KK = NB_K / KS;         // waves per tile, k rows per wave
    constexpr int NW = 27 * MT * NT * 256;                    // sums of a block
    constexpr int BUF = (NB_LC * SA + NB_OC * SG) / 8;
    constexpr int RED = (NW + MT * 16) / 4;
    __shared__ uint4 smem[2 * BUF > RED ? 2 * BUF : RED];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, row = lane & 15, kg = lane >> 4;
    const int mt = wave % MT, nt = (wave / MT) % NT, ks = wave / (MT * NT);
    const int nbi = (d.Ni + NB_I - 1) / NB_I, nbj = (d.Nj + NB_J - 1) / NB_J, nb = nbi * nbj * ((d.Nk + NB_K - 1) / NB_K);
    const int run = brick_run(nb), b0 = (blockIdx.x & 7) * run, b1 = min(b0 + run, nb), step = gridDim.x >> 3;
    uint4 v[NIT];
    auto fetch = [&](int b) {
        const int oi = NB_I * (b % nbi), oj = NB_J * ((b / nbi) % nbj), ok = NB_K * (b / (nbi * nbj));
#pragma unroll
        for (int it = 0; it < NIT; it++) {
            const int e = tid + 512 * it;
            v[it] = uint4{0u, 0u, 0u, 0u};
            if (e < NA) {          // as the convolutions: neighbours of the flattened index
                const int c = e / PA, li = c % NB_LI, lj = (c / NB_LI) % NB_LJ, lk = c / (NB_LI * NB_LJ);
                const int p = (oi - 1 + li) + d.Ni * ((oj - 1 + lj) + d.Nj * (ok - 1 + lk));
                if (p >= 0 && p < d.nc) v[it] = *reinterpret_cast<const uint4 *>(act + (size_t)p * NET_C + 8 * (e % PA));
            } else if (e < NA + NG) {
                const int c = (e - NA) / PG, i = oi + c % NB_I, j = oj + (c / NB_I) % NB_J, k = ok + c / (NB_I * NB_J);
                if (i < d.Ni && j < d.Nj && k < d.Nk)
                    v[it] = *reinterpret_cast<const uint4 *>(g + ((size_t)i + (size_t)d.Ni * (j + (size_t)d.Nj * k)) * NET_C + 8 * ((e - NA) % PG));
            }
        }
    };
    auto stage = [&](uint4 *buf) {
#pragma unroll
        for (int it = 0; it < NIT; it++) {
            const int e = tid + 512 * it;
            if (e < NA) buf[(e / PA) * (SA / 8) + e % PA] = v[it];
            else if (e < NA + NG) buf[NB_LC * SA / 8 + ((e - NA) / PG) * (SG / 8) + (e - NA) % PG] = v[it];
        }
    };
    const uint32_t o1 = 0x3F803F80u;   // two BF16 ones
    const uint4 o4 = {o1, o1, o1, o1};
    bf16x8 ones;
    memcpy(&ones, &o4, 16);
    f32x4 acc[27], accb = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int q = 0; q < 27; q++) acc[q] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int cell = 4 * kg + (row >> 2), ch = 4 * (row & 3);   // this lane's address in a transposing read
    int b = b0 + (blockIdx.x >> 3);
    if (b < b1) { fetch(b); stage(smem); }
    for (int cur = 0; b < b1; b += step, cur ^= 1) {
        __syncthreads();   // this brick staged; every wave is done with the other buffer
        const bool more = b + step < b1;
        if (more) fetch(b + step);
        const u16 *sA = reinterpret_cast<const u16 *>(smem + cur * BUF) + ((KK * ks) * (NB_LJ * NB_LI) + cell) * SA + 16 * nt + ch;
        const u16 *sG = reinterpret_cast<const u16 *>(smem + cur * BUF) + NB_LC * SA + ((KK * ks) * (NB_J * NB_I) + cell) * SG + 16 * mt + ch;
        bf16x8 av[KK][2];   // rows (s, s + 2) of the gradients
#pragma unroll
        for (int q = 0; q < 2 * KK; q++) {
            const u16 *r = sG + ((q / 2) * NB_J + q % 2) * NB_I * SG;
            av[q / 2][q % 2] = tr_rows(r, r + 2 * NB_I * SG);
        }
        if (nt == 0) {
#pragma unroll
            for (int q = 0; q < 2 * KK; q++) accb = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[q / 2][q % 2], ones, accb, 0, 0, 0);
        }
#pragma unroll
        for (int n = 0; n < (KK + 2) * 3; n++) {
            const int pl = n / 3, dx = n % 3;   // staged plane: dz = pl - k row (0..2)
            bf16x8 bv[4];                       // staged rows (x, x + 2): dy = x - s
#pragma unroll
            for (int x = 0; x < 4; x++) {
                const u16 *r = sA + ((pl * NB_LJ + x) * NB_LI + dx) * SA;
                bv[x] = tr_rows(r, r + 2 * NB_LI * SA);
            }
#pragma unroll
            for (int k = 0; k < KK; k++) {
                if (pl - k < 0 || pl - k > 2) continue;
#pragma unroll
                for (int q = 0; q < 6; q++) {
                    const int tap = 9 * (pl - k) + 3 * (q % 3) + dx;
                    acc[tap] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[k][q / 3], bv[q / 3 + q % 3], acc[tap], 0, 0, 0);
                }
            }
        }
        if (more) stage(smem + (cur ^ 1) * BUF);
    }
    // D[i = co][j = ci]: lane holds co = 16 mt + 4 kg + r, ci = 16 nt + row
    float *red = reinterpret_cast<float *>(smem);
    for (int q = 0; q < KS; q++) {
        __syncthreads();
        if (ks != q) continue;
#pragma unroll
        for (int t = 0; t < 27; t++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                float &x = red[((t * MT + mt) * 16 + 4 * kg + r) * (16 * NT) + 16 * nt + row];
                x = q == 0 ? acc[t][r] : x + acc[t][r];
            }
        if (nt == 0 && row == 0) {
#pragma unroll
            for (int r = 0; r < 4; r++) {
                float &x = red[NW + 16 * mt + 4 * kg + r];
                x = q == 0 ? accb[r] : x + accb[r];
            }
        }
    }
    __syncthreads();
    // workspace of a block: 27 taps of [co][ci], then the biases
    for (int e = tid; e < RED; e += 512) reinterpret_cast<uint4 *>(ws)[(size_t)blockIdx.x * RED + e] = smem[e];
}

// the blocks' sums onto the unpadded parameter layout [tap][nco][nci], [nco]: 64 sums per
// block, each in 16 runs of blocks added in order
template <int MT, int NT>
__global__ void __launch_bounds__(256) k_wreduce(const float *__restrict__ ws, int nblk, int nco, int nci, float *__restrict__ dW,
                                                 float *__restrict__ db) {
    constexpr int NW = 27 * MT * NT * 256, N = NW + MT * 16;
    __shared__ float part[16][64];
    const int run = (nblk + 15) / 16, q = threadIdx.x & 15, r = threadIdx.x >> 4;   // 4 sums, blocks [r run, (r + 1) run)
    const int e0 = blockIdx.x * 64 + 4 * q, b0 = r * run, b1 = min(b0 + run, nblk);
    float4 s = {0.f, 0.f, 0.f, 0.f};
    if (e0 < N) {
#pragma unroll 8
        for (int b = b0; b < b1; b++) {
            const float4 x = *reinterpret_cast<const float4 *>(ws + (size_t)b * N + e0);
            s.x += x.x; s.y += x.y; s.z += x.z; s.w += x.w;
        }
    }
    part[r][4 * q] = s.x; part[r][4 * q + 1] = s.y; part[r][4 * q + 2] = s.z; part[r][4 * q + 3] = s.w;
    __syncthreads();
    const int e = blockIdx.x * 64 + threadIdx.x;
    if (threadIdx.x >= 64 || e >= N) return;
    const int ci = e % (16 * NT), co = e < NW ? (e / (16 * NT)) % (16 * MT) : e - NW, tap = e / (MT * NT * 256);
    if (co >= nco || (e < NW && ci >= nci)) return;
    float t = 0.f;
#pragma unroll
    for (int k = 0; k < 16; k++) t += part[k][threadIdx.x];
    if (e < NW) dW[((size_t)tap * nco + co) * nci + ci] += t;
    else db[co] += t;
}

__device__ __forceinline__ uint4 pack8(const float (&f)[8]) {
    uint32_t o[4];
#pragma unroll
    for (int h = 0; h < 4; h++) o[h] = (uint32_t)f2bf(f[2 * h]) | ((uint32_t)f2bf(f[2 * h + 1]) << 16);
    return uint4{o[0], o[1], o[2], o[3]};
}
// dL/dout (FP32 [nc][8]) -> BF16 gradient of the last layer; zero outside the
// computed cells, where the output is not defined.  The cell's channels 8..31 are
// zeros (the buffer held another layer's gradient).
__global__ void __launch_bounds__(256) k_dout(NetDims d, const float *__restrict__ dout, u16 *__restrict__ g) {
    const int p = blockIdx.x * 256 + threadIdx.x;
    if (p >= d.nc) return;
    uint4 v = {0u, 0u, 0u, 0u};
    if (p >= d.lo && p < d.hi) {
        float f[8];
#pragma unroll
        for (int c = 0; c < 8; c++) f[c] = dout[(size_t)p * 8 + c];
        v = pack8(f);
    }
    uint4 *gp = reinterpret_cast<uint4 *>(g + (size_t)p * NET_C);
    gp[0] = v;
#pragma unroll
    for (int q = 1; q < 4; q++) gp[q] = uint4{0u, 0u, 0u, 0u};
}

// state -> input features ((rho - rho0)/s_rho, v/s_v, (p - p0)/s_p, B/s_B) of cell p
// from the cell's (rho, rho v, E, B) rounded to FP32 in q[8]
__device__ __forceinline__ void features_calc(const float (&q)[8], float gamma, float4 sc, float2 off, float (&f)[8]) {
    float rho = q[0], mx = q[1], my = q[2], mz = q[3];
    float E = q[4];
    float r = fmaxf(rho, 1e-12f);
    float vx = mx / r, vy = my / r, vz = mz / r;
    float P = (gamma - 1.f) * (E - 0.5f * r * (vx * vx + vy * vy + vz * vz));
    f[0] = (rho - off.x) / sc.x; f[1] = vx / sc.y; f[2] = vy / sc.y; f[3] = vz / sc.y; f[4] = (P - off.y) / sc.z;
    f[5] = q[5] / sc.w; f[6] = q[6] / sc.w; f[7] = q[7] / sc.w;
}
template <typename R>
__device__ __forceinline__ void state_of(size_t p, size_t n, const R *__restrict__ Gas, const R *__restrict__ B, float (&q)[8]) {
#pragma unroll
    for (int v = 0; v < 5; v++) q[v] = (float)Gas[v * n + p];
#pragma unroll
    for (int v = 0; v < 3; v++) q[5 + v] = (float)B[v * n + p];
}
template <typename R>
__device__ __forceinline__ void features_of(size_t p, size_t n, const R *__restrict__ Gas, const R *__restrict__ B, float gamma,
                                            float4 sc, float2 off, float (&f)[8]) {
    float q[8];
    state_of<R>(p, n, Gas, B, q);
    features_calc(q, gamma, sc, off, f);
}

// the features, BF16 (channels 8..31 stay the zeros of the allocation)
template <typename R>
__global__ void __launch_bounds__(256) k_features(int nc, const R *__restrict__ Gas, const R *__restrict__ B, float gamma,
                                                  float4 sc, float2 off, u16 *__restrict__ act) {
    int p = blockIdx.x * 256 + threadIdx.x;
    if (p >= nc) return;
    float f[8];
    features_of<R>(p, nc, Gas, B, gamma, sc, off, f);
    *reinterpret_cast<uint4 *>(act + (size_t)p * NET_C) = pack8(f);
}

// ----------------------------------------------------------------- inference
// One layer on bricks, as k_conv, but the layer's outputs are stored on a box
// [lo, lo + n) per axis only (the last layer's box is the cells at least `halo` from
// the grid faces, each earlier layer's box one cell wider on every side, so every
// stored output reads stored inputs); staged cells off the grid are zeros and feed
// only outputs that are not stored.  The first layer (CIN = 8) computes the
// features of its staged cells from Gas and B itself (as k_features).  Per
// output cell the operands, their K order, the bias and the activation are
// k_conv's, so the stored values equal gam_net_forward's bit for bit.
// The last layer alone on 134^3 cells: 103 us with weights fetched per brick -> 78.
struct InferBox { int lo[3], n[3], nb[3]; };

template <int CIN, int NCO, int MODE, typename R>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(CIN == 32 ? 2 : 4)))
k_infer(NetDims d, InferBox bx, const u16 *__restrict__ in, const R *__restrict__ Gas, const R *__restrict__ Bc, float gamma,
        float4 sc, float2 offs, const u16 *__restrict__ W, const float *__restrict__ bias, u16 *__restrict__ act_out,
        float *__restrict__ out) {
    static_assert(CIN == 8 || CIN == 32, "8 or 32 input channels");
    using T = ConvT<CIN, NCO>;
    constexpr int CS = T::CS, OS = T::OS, PER = CIN == 8 ? 1 : 4;
    constexpr int NIT = (NB_LC * PER + 255) / 256;
    __shared__ uint4 sIn[NB_LC * CS / 8];
    __shared__ uint4 sOut[MODE == 1 ? NB_OC * 2 : NB_OC * OS / 8];
    u16 *sO = reinterpret_cast<u16 *>(sOut);
    float *sF = reinterpret_cast<float *>(sOut);
    const int nbrick = bx.nb[0] * bx.nb[1] * bx.nb[2], run = brick_run(nbrick);
    const int b0 = (blockIdx.x & 7) * run, b1 = min(b0 + run, nbrick), step = gridDim.x >> 3;
    int b = b0 + (blockIdx.x >> 3);
    auto origin = [&](int bb, int &oi, int &oj, int &ok) {   // cell of the brick's box
        oi = NB_I * (bb % bx.nb[0]); oj = NB_J * ((bb / bx.nb[0]) % bx.nb[1]); ok = NB_K * (bb / (bx.nb[0] * bx.nb[1]));
    };
    // staged cell c: (origin - 1) + (li, lj, lk)
    auto cell_at = [&](int bb, int c, size_t &p) -> bool {
        int oi, oj, ok;
        origin(bb, oi, oj, ok);
        const int i = bx.lo[0] + oi - 1 + c % NB_LI, j = bx.lo[1] + oj - 1 + (c / NB_LI) % NB_LJ, k = bx.lo[2] + ok - 1 + c / (NB_LI * NB_LJ);
        p = (size_t)i + (size_t)d.Ni * ((size_t)j + (size_t)d.Nj * k);
        return i >= 0 && i < d.Ni && j >= 0 && j < d.Nj && k >= 0 && k < d.Nk;
    };
    uint4 v[CIN == 32 ? NIT : 1];
    float q8[CIN == 8 ? NIT : 1][8];
    bool live[NIT];
    auto fetch = [&](int bb) {
#pragma unroll
        for (int it = 0; it < NIT; it++) {
            const int e = threadIdx.x + 256 * it;
            size_t p = 0;
            live[it] = e < NB_LC * PER && cell_at(bb, e / PER, p);
            if constexpr (CIN == 8) {
                if (live[it]) state_of<R>(p, d.nc, Gas, Bc, q8[it]);
            } else {
                v[it] = uint4{0u, 0u, 0u, 0u};
                if (live[it]) v[it] = *reinterpret_cast<const uint4 *>(in + p * NET_C + 8 * (e % PER));
            }
        }
    };
    if (b >= b1) return;
    fetch(b);
    T cv;
    cv.init(W);
    for (; b < b1; b += step) {
#pragma unroll
        for (int it = 0; it < NIT; it++) {
            const int e = threadIdx.x + 256 * it;
            if (e >= NB_LC * PER) break;
            if constexpr (CIN == 8) {
                uint4 x = {0u, 0u, 0u, 0u};
                if (live[it]) {
                    float f[8];
                    features_calc(q8[it], gamma, sc, offs, f);
                    x = pack8(f);
                }
                sIn[e] = x;
            } else {
                sIn[(e / PER) * (CS / 8) + e % PER] = v[it];
            }
        }
        __syncthreads();   // staged; and every wave has read the last brick's sOut
        if (CIN == 32 && b + step < b1) fetch(b + step);
        cv.run(reinterpret_cast<const u16 *>(sIn));
#pragma unroll
        for (int q = 0; q < T::KT * NB_J * T::TW; q++) {
            const int kt = q / (NB_J * T::TW), m = (q / T::TW) % NB_J, t = q % T::TW;
            const int co = 16 * (cv.t0 + t) + cv.row, oc = ((cv.kr + kt) * NB_J + m) * NB_I + 4 * cv.kg;
            const f32x4 x = cv.acc[kt][m][t];
            if (MODE == 0 || co < 8) {
                const float bb = bias[co];
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const float y = x[r] + bb;
                    if constexpr (MODE == 0) sO[(oc + r) * OS + co] = f2bf(y > 0.f ? y : NET_LEAK * y);
                    else sF[(oc + r) * 8 + co] = y;
                }
            }
        }
        __syncthreads();   // results in sOut; and every wave is done with sIn
        int oi, oj, ok;
        origin(b, oi, oj, ok);
        constexpr int CH = MODE == 1 ? 2 : 4;   // 16-byte pieces per output cell
        for (int e = threadIdx.x; e < NB_OC * CH; e += 256) {
            const int oc = e / CH, part = e % CH;
            const int ii = oi + oc % NB_I, jj = oj + (oc / NB_I) % NB_J, kk = ok + oc / (NB_I * NB_J);
            if (ii >= bx.n[0] || jj >= bx.n[1] || kk >= bx.n[2]) continue;
            const size_t p = (size_t)(bx.lo[0] + ii) + (size_t)d.Ni * ((size_t)(bx.lo[1] + jj) + (size_t)d.Nj * (bx.lo[2] + kk));
            if constexpr (MODE == 0) *reinterpret_cast<uint4 *>(act_out + p * NET_C + 8 * part) = sOut[oc * (OS / 8) + part];
            else *reinterpret_cast<uint4 *>(out + p * 8 + 4 * part) = sOut[e];
        }
    }
}

// Adam on the FP32 master parameters (Kingma & Ba 2015, bias-corrected)
__global__ void __launch_bounds__(256) k_adam(int n, float *__restrict__ w, const float *__restrict__ g,
                                              float *__restrict__ m, float *__restrict__ v, float lr, float b1, float b2,
                                              float eps, float c1, float c2) {
    int q = blockIdx.x * 256 + threadIdx.x;
    if (q >= n) return;
    const float gq = g[q];
    const float mq = b1 * m[q] + (1.f - b1) * gq;
    const float vq = b2 * v[q] + (1.f - b2) * gq * gq;
    m[q] = mq;
    v[q] = vq;
    w[q] = w[q] - lr * (mq / c1) / (sqrtf(vq / c2) + eps);
}

// master FP32 parameters -> BF16 forward and transposed/flipped backward weights
// layer l forward: Wf[tap][co][ci]; backward data: Wb[tap'][ci][co] with tap' the mirrored tap
__global__ void __launch_bounds__(256) k_pack(const float *__restrict__ w, int off, int nco_real, int nci_real, int nco_pad,
                                              u16 *__restrict__ Wf, u16 *__restrict__ Wb) {
    int q = blockIdx.x * 256 + threadIdx.x;
    const int total = NET_TAPS * nco_pad * NET_C;
    if (q >= total) return;
    const int ci = q % NET_C, co = (q / NET_C) % nco_pad, tap = q / (NET_C * nco_pad);
    const float val = (co < nco_real && ci < nci_real) ? w[off + (tap * nco_real + co) * nci_real + ci] : 0.f;
    Wf[q] = f2bf(val);
    // backward data kernel has NCO = 32 outputs (= ci) and 32 inputs (= co, padded)
    const int mt = NET_TAPS - 1 - tap;
    if (ci < NET_C && co < NET_C) Wb[((size_t)mt * NET_C + ci) * NET_C + co] = f2bf(val);
}

// the first layer's weights, 4 taps per K step: W0[g][co][8q + ci] = w[tap = 4g + q][co][ci]
__global__ void __launch_bounds__(256) k_pack0(const float *__restrict__ w, u16 *__restrict__ W0) {
    const int q = blockIdx.x * 256 + threadIdx.x;
    if (q >= NET_G0 * NET_C * NET_C) return;
    const int k = q % NET_C, co = (q / NET_C) % NET_C, g = q / (NET_C * NET_C);
    const int tap = 4 * g + k / 8, ci = k % 8;
    W0[q] = tap < NET_TAPS ? f2bf(w[(tap * NET_C + co) * 8 + ci]) : (u16)0;
}

// ----------------------------------------------------------------- host side
struct gam_net {
    NetDims d;
    hipStream_t stream = nullptr;        // where the net's work goes: its own stream or the caller's
    hipStream_t own = nullptr;           // the stream the net created
    hipEvent_t done = nullptr;           // recorded after each gam_net_infer
    // parameters: FP32 master, grads, Adam moments
    float *w = nullptr, *g = nullptr, *m = nullptr, *v = nullptr;
    u16 *Wf[3] = {}, *Wb[3] = {};
    u16 *act[3] = {}, *inf[2] = {};      // forward: 0 features, 1..2 hidden; inference's hidden
                                         // (a backward pass takes the last forward's)
    u16 *gr[2] = {};                     // gradient ping-pong
    float *out = nullptr;
    float *dbuf = nullptr;               // upstream gradient uploaded from the host
    float *ws = nullptr;                 // the weight-gradient blocks' sums (k_wgrad)
    float4 scales = {1.f, 1.f, 1.f, 1.f};
    float gamma = 5.f / 3.f;
    float2 offs = {0.f, 0.f};
    std::string err;
};

// parameter layout (FP32): layer 0 W[27][32][8], b[32]; layer 1 W[27][32][32], b[32]; layer 2 W[27][8][32], b[8]
static const int kCo[3] = {32, 32, 8}, kCi[3] = {8, 32, 32}, kCoPad[3] = {32, 32, 16};
static int woff(int l) { int o = 0; for (int q = 0; q < l; q++) o += NET_TAPS * kCo[q] * kCi[q] + kCo[q]; return o; }
static int boff(int l) { return woff(l) + NET_TAPS * kCo[l] * kCi[l]; }

extern "C" int gam_net_num_params(void) { return woff(3); }

static int nfail(gam_net *n, int code, const char *msg, hipError_t e) {
    if (n) n->err = std::string(msg) + ": " + hipGetErrorString(e);
    return code;
}
#define NCHK(n, x) do { hipError_t e_ = (x); if (e_ != hipSuccess) return nfail(n, -2, #x, e_); } while (0)

extern "C" int gam_net_destroy(gam_net *n) {
    if (!n) return 0;
    if (n->own) (void)hipStreamSynchronize(n->own);   // work on a caller's stream: hipFree below waits for the device
    void *bufs[] = {n->w, n->g, n->m, n->v, n->out, n->dbuf, n->ws};
    for (void *b : bufs) if (b) (void)hipFree(b);
    for (int l = 0; l < 3; l++) { (void)hipFree(n->Wf[l]); (void)hipFree(n->Wb[l]); }
    for (u16 *b : {n->act[0], n->act[1], n->act[2], n->inf[0], n->inf[1], n->gr[0], n->gr[1]}) (void)hipFree(b);
    if (n->done) (void)hipEventDestroy(n->done);
    if (n->own) (void)hipStreamDestroy(n->own);
    delete n;
    return 0;
}

extern "C" int gam_net_create(int Ni, int Nj, int Nk, gam_net **out) {
    if (!out || Ni < 8 || Nj < 8 || Nk < 8) return -1;   // the 3-layer stencil needs 3 cells around each used cell
    *out = nullptr;
    long nc = (long)Ni * Nj * Nk;
    if ((nc + 28) * NET_C > 0x7fffffffL) return -1;
    gam_net *n = new gam_net();
    NetDims &d = n->d;
    d.Ni = Ni; d.Nj = Nj; d.Nk = Nk; d.nc = (int)nc;
    d.lo = Ni * Nj + Ni + 1;
    d.hi = d.nc - d.lo;
    auto cleanup = [&](int c) { gam_net_destroy(n); return c; };
    if (hipStreamCreateWithFlags(&n->own, hipStreamNonBlocking) != hipSuccess) return cleanup(-2);
    n->stream = n->own;
    if (hipEventCreateWithFlags(&n->done, hipEventDisableTiming) != hipSuccess) return cleanup(-2);
    const int np = gam_net_num_params();
    for (float **p : {&n->w, &n->g, &n->m, &n->v}) {
        if (hipMalloc(p, np * sizeof(float)) != hipSuccess) return cleanup(-3);
        if (hipMemset(*p, 0, np * sizeof(float)) != hipSuccess) return cleanup(-2);
    }
    for (int l = 0; l < 3; l++) {
        if (hipMalloc(&n->Wf[l], (size_t)NET_TAPS * kCoPad[l] * NET_C * 2) != hipSuccess) return cleanup(-3);
        if (hipMalloc(&n->Wb[l], (size_t)NET_TAPS * NET_C * NET_C * 2) != hipSuccess) return cleanup(-3);
        if (hipMemset(n->Wb[l], 0, (size_t)NET_TAPS * NET_C * NET_C * 2) != hipSuccess) return cleanup(-2);
    }
    const size_t ab = (size_t)nc * NET_C * 2;
    for (u16 **p : {&n->act[0], &n->act[1], &n->act[2], &n->inf[0], &n->inf[1], &n->gr[0], &n->gr[1]}) {
        if (hipMalloc(p, ab) != hipSuccess) return cleanup(-3);
        if (hipMemset(*p, 0, ab) != hipSuccess) return cleanup(-2);
    }
    if (hipMalloc(&n->out, (size_t)nc * 8 * sizeof(float)) != hipSuccess) return cleanup(-3);
    if (hipMalloc(&n->dbuf, (size_t)nc * 8 * sizeof(float)) != hipSuccess) return cleanup(-3);
    if (hipMalloc(&n->ws, (size_t)WG_BLOCKS * (27 * 1024 + 32) * sizeof(float)) != hipSuccess) return cleanup(-3);
    if (hipMemset(n->out, 0, (size_t)nc * 8 * sizeof(float)) != hipSuccess) return cleanup(-2);
    *out = n;
    return 0;
}

extern "C" const char *gam_net_error(const gam_net *n) { return n ? n->err.c_str() : "null net"; }
extern "C" void *gam_net_stream(gam_net *n) { return n ? (void *)n->stream : nullptr; }

extern "C" int gam_net_set_stream(gam_net *n, void *stream) {
    if (!n) return -1;
    hipStream_t to = stream ? (hipStream_t)stream : n->own;
    if (to == n->stream) return 0;
    NCHK(n, hipStreamSynchronize(n->stream));   // the work already queued ends before any on the new stream
    n->stream = to;
    return 0;
}
extern "C" const float *gam_net_output(gam_net *n) { return n ? n->out : nullptr; }
extern "C" float *gam_net_grad_buffer(gam_net *n) { return n ? n->dbuf : nullptr; }

static int pack(gam_net *n) {
    hipLaunchKernelGGL(k_pack0, dim3((NET_G0 * NET_C * NET_C + 255) / 256), 256, 0, n->stream, (const float *)n->w + woff(0),
                       n->Wf[0]);
    for (int l = 1; l < 3; l++) {
        const int total = NET_TAPS * kCoPad[l] * NET_C;
        hipLaunchKernelGGL(k_pack, dim3((total + 255) / 256), 256, 0, n->stream, (const float *)n->w, woff(l), kCo[l], kCi[l],
                           kCoPad[l], n->Wf[l], n->Wb[l]);
    }
    NCHK(n, hipGetLastError());
    return 0;
}

extern "C" int gam_net_set_params(gam_net *n, const float *w) {
    if (!n || !w) return -1;
    NCHK(n, hipMemcpyAsync(n->w, w, gam_net_num_params() * sizeof(float), hipMemcpyHostToDevice, n->stream));
    int rc = pack(n);
    if (rc) return rc;
    NCHK(n, hipStreamSynchronize(n->stream));
    return 0;
}

extern "C" int gam_net_get_params(gam_net *n, float *w, float *grad) {
    if (!n) return -1;
    if (w) NCHK(n, hipMemcpyAsync(w, n->w, gam_net_num_params() * sizeof(float), hipMemcpyDeviceToHost, n->stream));
    if (grad) NCHK(n, hipMemcpyAsync(grad, n->g, gam_net_num_params() * sizeof(float), hipMemcpyDeviceToHost, n->stream));
    NCHK(n, hipStreamSynchronize(n->stream));
    return 0;
}

extern "C" int gam_net_set_scales(gam_net *n, float rho, float v, float p, float b, float gamma) {
    if (!n || !(rho > 0) || !(v > 0) || !(p > 0) || !(b > 0)) return -1;
    n->scales = make_float4(rho, v, p, b);
    n->gamma = gamma;
    return 0;
}

extern "C" int gam_net_set_offsets(gam_net *n, float rho0, float p0) {
    if (!n) return -1;
    n->offs = make_float2(rho0, p0);
    return 0;
}

extern "C" int gam_net_features(gam_net *n, const void *Gas, const void *B, int precision) {
    if (!n || !Gas || !B) return -1;
    const int nb = (n->d.nc + 255) / 256;
    if (precision) hipLaunchKernelGGL(HIP_KERNEL_NAME(k_features<float>), dim3(nb), 256, 0, n->stream, n->d.nc, (const float *)Gas,
                                      (const float *)B, n->gamma, n->scales, n->offs, n->act[0]);
    else hipLaunchKernelGGL(HIP_KERNEL_NAME(k_features<double>), dim3(nb), 256, 0, n->stream, n->d.nc, (const double *)Gas,
                            (const double *)B, n->gamma, n->scales, n->offs, n->act[0]);
    NCHK(n, hipGetLastError());
    return 0;
}

extern "C" int gam_net_set_features(gam_net *n, const float *feat) {
    // host features [nc][8] FP32 (tests): rounded to BF16 like k_features
    if (!n || !feat) return -1;
    const size_t nc = n->d.nc;
    std::vector<u16> a(nc * NET_C, 0);
    for (size_t p = 0; p < nc; p++)
        for (int c = 0; c < 8; c++) a[p * NET_C + c] = f2bf(feat[p * 8 + c]);
    NCHK(n, hipMemcpyAsync(n->act[0], a.data(), a.size() * 2, hipMemcpyHostToDevice, n->stream));
    NCHK(n, hipStreamSynchronize(n->stream));
    return 0;
}

static unsigned conv_blocks(const gam_net *n, long most) {
    const NetDims &d = n->d;
    return brick_blocks((long)((d.Ni + NB_I - 1) / NB_I) * ((d.Nj + NB_J - 1) / NB_J) * ((d.Nk + NB_K - 1) / NB_K), most);
}
static dim3 conv_grid(const gam_net *n, int cin) { return dim3(conv_blocks(n, cin == 32 ? NB_STAY : 0x7fffffffL)); }

extern "C" int gam_net_forward(gam_net *n) {
    if (!n) return -1;
    const NetDims &d = n->d;
    hipLaunchKernelGGL(HIP_KERNEL_NAME(k_conv<8, 32, 0>), conv_grid(n, 8), 256, 0, n->stream, d, (const u16 *)n->act[0], (const u16 *)n->Wf[0],
                       (const float *)(n->w + boff(0)), (const u16 *)nullptr, n->act[1], (float *)nullptr);
    hipLaunchKernelGGL(HIP_KERNEL_NAME(k_conv<32, 32, 0>), conv_grid(n, 32), 256, 0, n->stream, d, (const u16 *)n->act[1], (const u16 *)n->Wf[1],
                       (const float *)(n->w + boff(1)), (const u16 *)nullptr, n->act[2], (float *)nullptr);
    hipLaunchKernelGGL(HIP_KERNEL_NAME(k_conv<32, 16, 1>), conv_grid(n, 32), 256, 0, n->stream, d, (const u16 *)n->act[2], (const u16 *)n->Wf[2],
                       (const float *)(n->w + boff(2)), (const u16 *)nullptr, (u16 *)nullptr, n->out);
    NCHK(n, hipGetLastError());
    return 0;
}

extern "C" int gam_net_infer(gam_net *n, const void *Gas, const void *B, int precision, int halo) {
    if (!n || !Gas || !B) return -1;
    const NetDims &d = n->d;
    const int N[3] = {d.Ni, d.Nj, d.Nk};
    if (halo < 3) { n->err = "gam_net_infer: halo must be >= 3 (three layers of 3-point stencils)"; return -1; }
    for (int a = 0; a < 3; a++)
        if (N[a] < 2 * halo + 1) { n->err = "gam_net_infer: the grid is thinner than 2*halo + 1 cells"; return -1; }
    InferBox bx[3];
    for (int l = 0; l < 3; l++) {   // layer l stores the cells at least halo - (2 - l) from the faces
        const int lo = halo - (2 - l);
        const int nb[3] = {NB_I, NB_J, NB_K};
        for (int a = 0; a < 3; a++) {
            bx[l].lo[a] = lo;
            bx[l].n[a] = N[a] - 2 * lo;
            bx[l].nb[a] = (bx[l].n[a] + nb[a] - 1) / nb[a];
        }
    }
    u16 *h1 = n->inf[0], *h2 = n->inf[1];
    auto grid = [](int cin, const InferBox &b) { return dim3(brick_blocks((long)b.nb[0] * b.nb[1] * b.nb[2], cin == 32 ? NB_STAY : 0x7fffffffL)); };
    if (precision)
        hipLaunchKernelGGL(HIP_KERNEL_NAME(k_infer<8, 32, 0, float>), grid(8, bx[0]), 256, 0, n->stream, d, bx[0], (const u16 *)nullptr,
                           (const float *)Gas, (const float *)B, n->gamma, n->scales, n->offs, (const u16 *)n->Wf[0],
                           (const float *)(n->w + boff(0)), h1, (float *)nullptr);
    else
        hipLaunchKernelGGL(HIP_KERNEL_NAME(k_infer<8, 32, 0, double>), grid(8, bx[0]), 256, 0, n->stream, d, bx[0], (const u16 *)nullptr,
                           (const double *)Gas, (const double *)B, n->gamma, n->scales, n->offs, (const u16 *)n->Wf[0],
                           (const float *)(n->w + boff(0)), h1, (float *)nullptr);
    hipLaunchKernelGGL(HIP_KERNEL_NAME(k_infer<32, 32, 0, float>), grid(32, bx[1]), 256, 0, n->stream, d, bx[1], (const u16 *)h1,
                       (const float *)nullptr, (const float *)nullptr, n->gamma, n->scales, n->offs, (const u16 *)n->Wf[1],
                       (const float *)(n->w + boff(1)), h2, (float *)nullptr);
    hipLaunchKernelGGL(HIP_KERNEL_NAME(k_infer<32, 16, 1, float>), grid(32, bx[2]), 256, 0, n->stream, d, bx[2], (const u16 *)h2,
                       (const float *)nullptr, (const float *)nullptr, n->gamma, n->scales, n->offs, (const u16 *)n->Wf[2],
                       (const float *)(n->w + boff(2)), (u16 *)nullptr, n->out);
    NCHK(n, hipGetLastError());
    NCHK(n, hipEventRecord(n->done, n->stream));
    return 0;
}

extern "C" void *gam_net_infer_event(gam_net *n) { return n ? (void *)n->done : nullptr; }

// dout: device FP32 [nc][8] = dL/d(out).  Accumulates into the gradient buffer
// (gam_net_zero_grad clears it).  Uses the activations of the last forward.
extern "C" int gam_net_backward(gam_net *n, const float *dout) {
    if (!n || !dout) return -1;
    const NetDims &d = n->d;
    const dim3 wb(conv_blocks(n, WG_BLOCKS));
    auto wgrad = [&](auto mt, auto nt, const u16 *g, const u16 *a, int l) {
        constexpr int MT = decltype(mt)::value, NT = decltype(nt)::value;
        hipLaunchKernelGGL(HIP_KERNEL_NAME(k_wgrad<MT, NT>), wb, 512, 0, n->stream, d, g, a, n->ws);
        hipLaunchKernelGGL(HIP_KERNEL_NAME(k_wreduce<MT, NT>), dim3((27 * MT * NT * 256 + MT * 16 + 63) / 64), 256, 0, n->stream,
                           (const float *)n->ws, (int)wb.x, kCo[l], kCi[l], n->g + woff(l), n->g + boff(l));
    };
    const std::integral_constant<int, 1> one;
    const std::integral_constant<int, 2> two;
    hipLaunchKernelGGL(k_dout, dim3((d.nc + 255) / 256), 256, 0, n->stream, d, dout, n->gr[0]);
    // layer 2 (linear, 8 outputs padded to 16)
    wgrad(one, two, n->gr[0], n->act[2], 2);
    hipLaunchKernelGGL(HIP_KERNEL_NAME(k_conv<32, 32, 2>), conv_grid(n, 32), 256, 0, n->stream, d, (const u16 *)n->gr[0], (const u16 *)n->Wb[2],
                       (const float *)nullptr, (const u16 *)n->act[2], n->gr[1], (float *)nullptr);
    // layer 1
    wgrad(two, two, n->gr[1], n->act[1], 1);
    hipLaunchKernelGGL(HIP_KERNEL_NAME(k_conv<32, 32, 2>), conv_grid(n, 32), 256, 0, n->stream, d, (const u16 *)n->gr[1], (const u16 *)n->Wb[1],
                       (const float *)nullptr, (const u16 *)n->act[1], n->gr[0], (float *)nullptr);
    // layer 0 (input gradient not needed)
    wgrad(two, one, n->gr[0], n->act[0], 0);
    NCHK(n, hipGetLastError());
    return 0;
}

extern "C" int gam_net_zero_grad(gam_net *n) {
    if (!n) return -1;
    NCHK(n, hipMemsetAsync(n->g, 0, gam_net_num_params() * sizeof(float), n->stream));
    return 0;
}

extern "C" int gam_net_adam(gam_net *n, float lr, float b1, float b2, float eps, int t) {
    if (!n || t < 1) return -1;
    const int np = gam_net_num_params();
    const float c1 = 1.f - powf(b1, (float)t), c2 = 1.f - powf(b2, (float)t);
    hipLaunchKernelGGL(k_adam, dim3((np + 255) / 256), 256, 0, n->stream, np, n->w, (const float *)n->g, n->m, n->v, lr, b1, b2,
                       eps, c1, c2);
    NCHK(n, hipGetLastError());
    return pack(n);
}

extern "C" int gam_net_sync(gam_net *n) {
    if (!n) return -1;
    NCHK(n, hipStreamSynchronize(n->stream));
    return 0;
}

extern "C" int gam_net_get_output(gam_net *n, float *out) {
    if (!n || !out) return -1;
    NCHK(n, hipMemcpyAsync(out, n->out, (size_t)n->d.nc * 8 * sizeof(float), hipMemcpyDeviceToHost, n->stream));
    NCHK(n, hipStreamSynchronize(n->stream));
    return 0;
}

// channels-last BF16 activations of the last forward (layer 0 = features), for tests
extern "C" int gam_net_get_act(gam_net *n, int layer, unsigned short *out) {
    if (!n || !out || layer < 0 || layer > 2) return -1;
    NCHK(n, hipMemcpyAsync(out, n->act[layer], (size_t)n->d.nc * NET_C * 2, hipMemcpyDeviceToHost, n->stream));
    NCHK(n, hipStreamSynchronize(n->stream));
    return 0;
}

extern "C" int gam_net_backward_host(gam_net *n, const float *dout) {
    if (!n || !dout) return -1;
    NCHK(n, hipMemcpyAsync(n->dbuf, dout, (size_t)n->d.nc * 8 * sizeof(float), hipMemcpyHostToDevice, n->stream));
    return gam_net_backward(n, n->dbuf);
}
