// q4mm.hip - the dense Q4_0 products behind rvh_q4_mm, rvh_q4_mv (runtime/hip/rvhip.h:42-48) and
// rvm_q4_mm_n: Q4_0 rows in the reference layout (18-byte blocks: f16 d, 16 nibble bytes;
// runtime/src/ops.rs:83-92) times f32 activations. The reference's CPU ops are the tolerance target
// (runtime/tests/hip_ops.rs:56-81).
//
// Arithmetic under 16,384 rows, the same for every kernel (from there: k_q4_mm_i8, below), so that a token's
// result depends neither on the other tokens of the call nor on the launch shape (hip_ops.rs:73-78):
//  - a row's nb blocks fall into four parts of q4_part(nb) blocks;
//  - the token's activations of a block are scaled by 2^(141 - E), E the largest biased exponent of the
//    part's blocks up to this one (so that the largest lies under 2^15), or the block's own where that is
//    more than Q4_NEAR lower (q4_exponent), and split into two f16, each rounded: 2^-23 of the element or
//    of the block's largest;
//  - n - 8 is exact in f16, so v_mfma_f32_16x16x32_f16 sums exact products over one block: the low
//    halves first, the high halves onto them;
//  - acc = fma(d, sum, acc) in block order from 0; where E changes, acc is first scaled to the new one;
//  - the parts' sums, scaled back, add as (P0 + P1) + (P2 + P3).
// A non-finite activation makes the token's results NaN.
//
// The K order of a block in the MFMA: K group g (lanes 16 g ..) holds elements 4g, 4g + 2, 16 + 4g,
// 16 + 4g + 2, 4g + 1, 4g + 3, 16 + 4g + 1, 16 + 4g + 3, as the nibbles of dword g of the block come out
// of a mask (q4_f16). A holds the tokens as rows, B the weight rows as columns: lane (j, g) = (lane & 15,
// lane >> 4) receives tokens 4g .. 4g + 3 of weight row j.
#include "internal.hpp"

namespace rvm {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

template <int NW>
struct __attribute__((packed, aligned(2))) Q4Nibbles {
    uint32_t q[NW];
};
template <int N>
struct __attribute__((packed, aligned(4))) Dwords {
    uint32_t q[N];
};
struct __attribute__((packed, aligned(4))) Floats4 {
    float v[4];
};

constexpr int Q4_PARTS = 4;
// Blocks per part: even, so that the parts of a row whose blocks pair up on dwords start on a pair.
__host__ __device__ constexpr int q4_part(int nb) { return 2 * ((nb + 2 * Q4_PARTS - 1) / (2 * Q4_PARTS)); }

// The nibble masks and f16 biases, unknown to the compiler where it would otherwise make two
// instructions of a masked or.
struct Q4Masks {
    uint32_t lo = 0x000F000Fu, hi = 0x00F000F0u, one = 0x64006400u;
    __device__ __forceinline__ Q4Masks() {
        asm("" : "+s"(lo), "+s"(hi));
        asm("" : "+v"(one));
    }
};
// Eight nibbles n of a dword as n - 8 in f16: 0x6400 | n is 1024 + n, 0x6400 | 16 n is 1024 + 16 n.
__device__ __forceinline__ f16x8 q4_f16(uint32_t w, const Q4Masks &k) {
    const f16x2 b = {(_Float16)1032.0f, (_Float16)1032.0f}, s = {(_Float16)0.0625f, (_Float16)0.0625f},
                t = {(_Float16)-72.0f, (_Float16)-72.0f};
    const uint32_t v = w >> 8;
    return as_f16x8(as_u32(as_f16x2((w & k.lo) | k.one) - b),
                    as_u32(__builtin_elementwise_fma(as_f16x2((w & k.hi) | k.one), s, t)),
                    as_u32(as_f16x2((v & k.lo) | k.one) - b),
                    as_u32(__builtin_elementwise_fma(as_f16x2((v & k.hi) | k.one), s, t)));
}

// split2_f16 with the pairs as dwords
__device__ __forceinline__ void q4_split(float x0, float x1, uint32_t &hi, uint32_t &lo) {
    f16x2 h, l;
    split2_f16(x0, x1, h, l);
    hi = as_u32(h);
    lo = as_u32(l);
}

// Lane rows of 16: after swap32, a = (a's rows 0 1, b's 0 1), b = (a's 2 3, b's 2 3); after swap16,
// a = (a0, b0, a2, b2), b = (a1, b1, a3, b3).
__device__ __forceinline__ void swap32(uint32_t &a, uint32_t &b) {
    const u32x2 r = __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane32_swap(a, b, false, false));
    a = r.x;
    b = r.y;
}
__device__ __forceinline__ void swap16(uint32_t &a, uint32_t &b) {
    const u32x2 r = __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane16_swap(a, b, false, false));
    a = r.x;
    b = r.y;
}
// v[i] of lane row g becomes v[g] of lane row i
__device__ __forceinline__ void rows_transpose(uint32_t (&v)[4]) {
    swap32(v[0], v[2]);
    swap32(v[1], v[3]);
    swap16(v[0], v[1]);
    swap16(v[2], v[3]);
}
// v[i] in every lane row: s of lane row i
__device__ __forceinline__ void rows_gather(uint32_t s, uint32_t (&v)[4]) {
    v[0] = v[2] = s;
    swap32(v[0], v[2]);
    v[1] = v[0];
    v[3] = v[2];
    swap16(v[0], v[1]);
    swap16(v[2], v[3]);
}

__device__ __forceinline__ int exp_field(float m) { return (int)((__float_as_uint(m) >> 23) & 0xFF); }

// The exponent that a block's activations are scaled by: own is the block's largest (0: zeros, whose scale
// does not matter, and subnormal values), top the part's largest up to it. A block far below top would keep
// few of its bits under top's scale, which a row needs whose weights of the large blocks are as much smaller
// than this one's, or zeros. 60 below top it stays: the sums so far must not pass the largest float.
constexpr int Q4_NEAR = 16, Q4_FAR = 60;
__device__ __forceinline__ int q4_exponent(int own, int top) {
    return own == 0 || own >= top - Q4_NEAR ? top : max(own, top - Q4_FAR);
}

// rows of an even block count on a 4-byte aligned matrix: every pair of blocks starts on a dword
__host__ __device__ __forceinline__ bool q4_rows_aligned(const uint8_t *w, int nb) {
    return (nb & 1) == 0 && ((uintptr_t)w & 3) == 0;
}

// Up to four matrices on one input in one launch: workgroups start[m] .. start[m + 1] - 1 take matrix m.
constexpr int Q4_NMAT = 4;
struct Q4Mats {
    const uint8_t *w[Q4_NMAT];
    float *y[Q4_NMAT];
    int n_out[Q4_NMAT];
    int start[Q4_NMAT + 1];  // start[n]: the workgroups in all
    int n;
};
// The workgroup's matrix. Every field is read at a fixed offset, so that all the kernel arguments come in
// one round trip (an index into the arrays made it two).
struct Q4Mat {
    const uint8_t *w;
    float *y;
    int n_out, wg;  // wg: the workgroup within the matrix
};
__device__ __forceinline__ Q4Mat q4_matrix(const Q4Mats &mats, int bx) {
    Q4Mat r = {mats.w[0], mats.y[0], mats.n_out[0], bx};
#pragma unroll
    for (int i = 1; i < Q4_NMAT; ++i) {
        const bool in = i < mats.n && bx >= mats.start[i];
        r.w = in ? mats.w[i] : r.w;
        r.y = in ? mats.y[i] : r.y;
        r.n_out = in ? mats.n_out[i] : r.n_out;
        r.wg = in ? bx - mats.start[i] : r.wg;
    }
    return r;
}

// ---- Up to four tokens. A workgroup of four waves takes 16 rows, wave p part p; lane (j, g) loads blocks
// 2g and 2g + 1 of every 8 of its row (36 bytes), all of a part's up to QV_CH passes at once, and the
// lane rows exchange the nibble dwords into the MFMA's order. The wave converts its own blocks of x
// while the weights are in flight (8 lanes per block) and reads them back from LDS, lane j token j's.
// Every load is unconditional (past the part: its last blocks again for the weights, zeros for x), so
// that each wait counts only what it needs. What bounds it: the launch, one round trip to HBM and the
// part's chain of blocks (one layer's seven projections in four launches of a graph: 23.1 us for one token,
// 24.0 with f32 products on the VALU; 4 tokens 29.8 / 41.5; loads under branches took 25.1).
constexpr int QV_CH = 4;  // passes of 8 blocks in registers at most

// How a lane loads its two blocks: as two, where the matrix starts on 2 bytes or its rows are one block; as 9
// dwords, where every pair starts on one; shifted, as the dwords that hold the 36 bytes (a pair 2 bytes past a
// dword ends in the low half of the last one, which is loaded as such). Two blocks at 2-byte addresses cost a
// row of 65 blocks half a microsecond and more (1 token, 1000 x 2080: 5.3 us, shifted 5.1; one layer's seven
// projections on odd block counts 29.2 / 26.6).
enum { QV_SPLIT, QV_DWORDS, QV_SHIFTED };

template <int NT, int NP, int LD>  // tokens a pass (blockIdx.y); the part's passes of 8 blocks, at most QV_CH at once
__global__ __launch_bounds__(64 * Q4_PARTS) void k_q4_vec(Q4Mats mats, const float *__restrict__ x, int k, int n_in) {
    __shared__ __attribute__((aligned(16))) uint32_t xs[Q4_PARTS][NT][NP * 8 * 32];  // [block][hi, lo][g][4]
    __shared__ float ps[Q4_PARTS][NT][16];
    const int lane = threadIdx.x & 63, j = lane & 15, g = lane >> 4;
    const int p = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const Q4Mat mat = q4_matrix(mats, blockIdx.x);
    const int n_out = mat.n_out, r0 = mat.wg * 16, t0 = blockIdx.y * NT;
    x += (size_t)t0 * k;
    n_in -= t0;
    const int nb = k / QK, qb = q4_part(nb), b0 = p * qb, b1 = min(nb, b0 + qb);
    const uint8_t *wr = mat.w + (size_t)min(r0 + j, n_out - 1) * ((size_t)nb * Q4_BLOCK);
    const Q4Masks km;
    float acc[NT];
    int E[NT], top[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        acc[t] = 0.0f;
        E[t] = top[t] = 1;
    }
    for (int c0 = b0; c0 < b1; c0 += 8 * NP) {
        // the activations' loads first (the weights' come from further away), then the weights'
        float4 xv[NP][NT];
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const __amdgpu_buffer_rsrc_t xrs = buffer_rsrc(x + (size_t)min(t, n_in - 1) * k, (uint32_t)b1 * QK * 4);
#pragma unroll
            for (int u = 0; u < NP; ++u)
                xv[u][t] = buffer_load4(xrs, (uint32_t)((c0 + 8 * u) * QK + 4 * lane) * 4, 0);
        }
        uint32_t v[NP][10];
#pragma unroll
        for (int u = 0; u < NP; ++u) {
            const int b = c0 + 8 * u + 2 * g;
            if constexpr (LD != QV_SPLIT) {
                const uint8_t *p = wr + min(b, nb - 2) * Q4_BLOCK;
                const uint8_t *a = LD == QV_SHIFTED ? (const uint8_t *)((uintptr_t)p & ~(uintptr_t)3) : p;
                const Dwords<4> d0 = *(const Dwords<4> *)a, d1 = *(const Dwords<4> *)(a + 16);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    v[u][i] = d0.q[i];
                    v[u][4 + i] = d1.q[i];
                }
                v[u][8] = *(const uint32_t *)(a + 32);
                if constexpr (LD == QV_SHIFTED) v[u][9] = *(const uint16_t *)(p + 34);
            } else {
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const uint8_t *a = wr + min(b + h, nb - 1) * Q4_BLOCK;
                    const Q4Nibbles<4> q = *(const Q4Nibbles<4> *)(a + 2);
                    v[u][5 * h] = *(const uint16_t *)a;
#pragma unroll
                    for (int i = 0; i < 4; ++i) v[u][5 * h + 1 + i] = q.q[i];
                }
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        // x: lane l takes elements 4 (l % 8) .. + 3 of block l / 8 of each pass
        int ev[NP][NT], own[NP][NT];  // the largest exponent up to this lane's block, and the block's
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int u = 0; u < NP; ++u) {
                const float4 f = xv[u][t];
                float mx = fmaxf(fmaxf(fabsf(f.x), fabsf(f.y)), fmaxf(fabsf(f.z), fabsf(f.w)));
                mx = maxf_bits(mx, dpp<0xb1>(__builtin_bit_cast(uint32_t, mx)));
                mx = maxf_bits(mx, dpp<0x4e>(__builtin_bit_cast(uint32_t, mx)));
                mx = maxf_bits(mx, dpp<0x141>(__builtin_bit_cast(uint32_t, mx)));
                own[u][t] = exp_field(mx);
                int e = max(own[u][t], top[t]);  // over the 8 blocks of the pass, then those before
                e = max(e, __builtin_amdgcn_update_dpp(0, e, 0x118, 0xf, 0xf, false));  // row_shr:8
                e = max(e, __builtin_amdgcn_update_dpp(0, e, 0x142, 0xa, 0xf, false));  // row_bcast:15
                ev[u][t] = max(e, __builtin_amdgcn_update_dpp(0, e, 0x143, 0xc, 0xf, false));  // row_bcast:31
            }
        wave_lds_sync();
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            if (c0 == b0) E[t] = __builtin_amdgcn_readlane(ev[0][t], 0);  // nothing to rescale yet
#pragma unroll
            for (int u = 0; u < NP; ++u) {
                if (u > 0) ev[u][t] = max(ev[u][t], top[t]);
                top[t] = __builtin_amdgcn_readlane(ev[u][t], 63);
                ev[u][t] = q4_exponent(own[u][t], ev[u][t]);
                const int s = 141 - ev[u][t];
                const float4 f = xv[u][t];
                uint32_t h0, l0, h1, l1;  // elements 0 and 2, 1 and 3
                q4_split(ldexpf(f.x, s), ldexpf(f.z, s), h0, l0);
                q4_split(ldexpf(f.y, s), ldexpf(f.w, s), h1, l1);
                uint32_t *d = xs[p][t] + (8 * u + (lane >> 3)) * 32 + (lane & 3) * 4 + ((lane >> 2) & 1);
                d[0] = h0;
                d[2] = h1;
                d[16] = l0;
                d[18] = l1;
            }
        }
        wave_lds_sync();
        const uint32_t *xr = xs[p][NT > 1 ? min(j, NT - 1) : 0] + 4 * g;
#pragma unroll
        for (int u = 0; u < NP; ++u) {
            if (c0 + 8 * u >= b1) break;
            uint32_t nib[2][4], ds[4], s;
            if constexpr (LD != QV_SPLIT) {
                if constexpr (LD == QV_SHIFTED) {
                    const uint32_t by = (uintptr_t)(wr + min(c0 + 8 * u + 2 * g, nb - 2) * Q4_BLOCK) & 2;
#pragma unroll
                    for (int i = 0; i < 9; ++i) v[u][i] = __builtin_amdgcn_alignbyte(v[u][i + 1], v[u][i], by);
                }
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    nib[0][i] = __builtin_amdgcn_perm(v[u][i + 1], v[u][i], 0x05040302u);
                    nib[1][i] = v[u][5 + i];
                }
                s = __builtin_amdgcn_perm(v[u][4], v[u][0], 0x07060100u);
                if (LD == QV_SHIFTED && c0 + 8 * u + 2 * g == nb - 1) {  // a row's last block, loaded behind another
#pragma unroll
                    for (int i = 0; i < 4; ++i) nib[0][i] = nib[1][i];
                    s >>= 16;
                }
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    nib[0][i] = v[u][1 + i];
                    nib[1][i] = v[u][6 + i];
                }
                s = v[u][0] | v[u][5] << 16;
            }
            // a block past the part weighs nothing, whatever it holds
            if (c0 + 8 * u + 2 * g >= b1) s &= 0xFFFF0000u;
            if (c0 + 8 * u + 2 * g + 1 >= b1) s &= 0x0000FFFFu;
            rows_transpose(nib[0]);
            rows_transpose(nib[1]);
            rows_gather(s, ds);
            // the pass's blocks, with a look at the exponents before each where one changes inside the pass
            auto pass = [&](auto changec) {
#pragma unroll
                for (int i0 = 0; i0 < 8; i0 += 4) {
                    f16x8 xh[4], wf[4];
                    f32x4 c[4];
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const uint4 *xq = (const uint4 *)(xr + (8 * u + i0 + i) * 32);
                        xh[i] = __builtin_bit_cast(f16x8, xq[0]);
                        wf[i] = q4_f16(nib[i & 1][(i0 + i) >> 1], km);
                        c[i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, xq[4]), wf[i],
                                                                      f32x4{0, 0, 0, 0}, 0, 0, 0);
                    }
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        c[i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xh[i], wf[i], c[i], 0, 0, 0);
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        if constexpr (decltype(changec)::value)
#pragma unroll
                            for (int t = 0; t < NT; ++t) {
                                const int e = __builtin_amdgcn_readlane(ev[u][t], 8 * (i0 + i));
                                acc[t] = ldexpf(acc[t], E[t] - e);
                                E[t] = e;
                            }
                        const f16x2 d = as_f16x2(ds[(i0 + i) >> 1]);
#pragma unroll
                        for (int t = 0; t < NT; ++t) acc[t] = fmaf((float)(i & 1 ? d.y : d.x), c[i][t], acc[t]);
                    }
                }
            };
            bool change = false;
#pragma unroll
            for (int t = 0; t < NT; ++t) change |= __builtin_amdgcn_ballot_w64(ev[u][t] != E[t]) != 0;
            if (change) pass(std::true_type{});
            else pass(std::false_type{});
        }
    }
    if (g == 0)  // tokens 0 .. 3 of the MFMA's rows
#pragma unroll
        for (int t = 0; t < NT; ++t) ps[p][t][j] = ldexpf(acc[t], E[t] - 141);
    __syncthreads();
    const int r = threadIdx.x & 15, t = threadIdx.x >> 4;
    if (t < NT && t < n_in && r0 + r < n_out)
        mat.y[(size_t)(t0 + t) * n_out + r0 + r] = (ps[0][t][r] + ps[1][t][r]) + (ps[2][t][r] + ps[3][t][r]);
}

// ---- Several tokens. A workgroup of four waves takes 16 RT rows x 16 TT tokens, wave p part p of the
// blocks; the waves meet only in the final sum. Lane (j, g) loads block g of every 4 of its rows (the
// next 4 while these are computed) and its 8 elements of each block of x of token j (PB blocks ahead).
// What bounds it, 8 x 2 tiles: VALU, about 250 instructions a wave and block (64 the folds, 72 the nibbles,
// 66 x, 32 the MFMAs), at 45% of its rate; without the loads 183 us where 265 are taken. One layer's seven
// projections of 512 tokens in four launches: 265 us (203 TFLOP/s) against 2,500 for f32 products on the
// VALU; 100 tokens 100 / 512, 16 tokens 48 / 98. Eight parts and eight waves a workgroup took 316 us (one
// workgroup per CU), 64 rows a wave throughout 305.
template <int RT, int TT, int PB>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void k_q4_tile(
    Q4Mats mats, const float *__restrict__ x, int k, int n_in) {
    __shared__ float4 ps[Q4_PARTS][RT][TT][64];
    const int lane = threadIdx.x & 63, j = lane & 15, g = lane >> 4;
    const int p = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if ((int)blockIdx.x >= mats.start[mats.n]) return;  // the grid's width is a multiple of the XCDs
    const Q4Mat mat = q4_matrix(mats, blockIdx.x);
    const int n_out = mat.n_out, r0 = mat.wg * 16 * RT, t0 = blockIdx.y * 16 * TT;
    const int nb = k / QK, qb = q4_part(nb), b0 = p * qb, b1 = min(nb, b0 + qb);
    const size_t rb = (size_t)nb * Q4_BLOCK;
    const uint8_t *wr[RT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) wr[rt] = mat.w + (size_t)min(r0 + 16 * rt + j, n_out - 1) * rb;
    const float *xr[TT];
#pragma unroll
    for (int tt = 0; tt < TT; ++tt) xr[tt] = x + (size_t)min(t0 + 16 * tt + j, n_in - 1) * k + 4 * g;

    const Q4Masks km;
    f32x4 acc[RT][TT];
    // token j's exponent, and what a float in [2^-16, 2) times its power of two exceeds by less than 17 << 23 as
    // bits; where E is a far block's, a value that every float exceeds by more, with the part's largest exponent
    // in its low byte
    int E[TT];
    uint32_t low[TT];
#pragma unroll
    for (int tt = 0; tt < TT; ++tt) {
        E[tt] = 1;
        low[tt] = (uint32_t)(1 - Q4_NEAR) << 23;
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) acc[rt][tt] = f32x4{0, 0, 0, 0};
    }
    uint32_t wn[RT][4], sn[RT];  // the next 4 blocks: block g of them, as loaded
    auto load_w = [&](int b, int rt) {
        const uint8_t *a = wr[rt] + min(b + g, nb - 1) * Q4_BLOCK;
        const Q4Nibbles<4> q = *(const Q4Nibbles<4> *)(a + 2);
        sn[rt] = *(const uint16_t *)a;
#pragma unroll
        for (int i = 0; i < 4; ++i) wn[rt][i] = q.q[i];
    };
    Floats4 xb[PB][TT][2];  // block b's at (b - b0) % PB
    auto load_x = [&](int b, int i, int tt) {
        const float *a = xr[tt] + (size_t)min(b, nb - 1) * QK;
        xb[i][tt][0] = *(const Floats4 *)a;
        xb[i][tt][1] = *(const Floats4 *)(a + 16);
    };
    if (b0 < b1) {
#pragma unroll
        for (int i = 0; i < PB; ++i)
#pragma unroll
            for (int tt = 0; tt < TT; ++tt) load_x(b0 + i, i, tt);
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) load_w(b0, rt);
    }
    for (int c0 = b0; c0 < b1; c0 += 4) {
        uint32_t nib[RT][4], ds[RT / 2][4];  // the scales of row tiles 2 i and 2 i + 1 in one dword
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
#pragma unroll
            for (int i = 0; i < 4; ++i) nib[rt][i] = wn[rt][i];
            rows_transpose(nib[rt]);
            if (rt % 2) rows_gather(sn[rt - 1] | sn[rt] << 16, ds[rt / 2]);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int b = c0 + i;
            if (b >= b1) break;
            // x of the block: its largest against the token's exponent, then the split
            f16x8 xh[TT], xl[TT];
#pragma unroll
            for (int tt = 0; tt < TT; ++tt) {
                const float *lo = xb[i % PB][tt][0].v, *hi = xb[i % PB][tt][1].v;
                float mx = fmaxf(fmaxf(fmaxf(fabsf(lo[0]), fabsf(lo[1])), fmaxf(fabsf(lo[2]), fabsf(lo[3]))),
                                 fmaxf(fmaxf(fabsf(hi[0]), fabsf(hi[1])), fmaxf(fabsf(hi[2]), fabsf(hi[3]))));
                if (__builtin_amdgcn_ballot_w64(__float_as_uint(mx) - low[tt] >= (Q4_NEAR + 1u) << 23)) {
                    mx = fmaxf(mx, __shfl_xor(mx, 16));
                    mx = fmaxf(mx, __shfl_xor(mx, 32));
                    const int own = exp_field(mx), far = low[tt] & 0xFF, top = max(far ? far : E[tt], own);
                    const int e = q4_exponent(own, top), change = E[tt] - e;
                    E[tt] = e;
                    low[tt] = e == top ? (uint32_t)(e - Q4_NEAR) << 23 : 0x80000000u | (uint32_t)top;
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int by = __shfl(change, 4 * g + r);
#pragma unroll
                        for (int rt = 0; rt < RT; ++rt) acc[rt][tt][r] = ldexpf(acc[rt][tt][r], by);
                    }
                }
                const int s = 141 - E[tt];
                uint32_t h[4], l[4];
                q4_split(ldexpf(lo[0], s), ldexpf(lo[2], s), h[0], l[0]);
                q4_split(ldexpf(hi[0], s), ldexpf(hi[2], s), h[1], l[1]);
                q4_split(ldexpf(lo[1], s), ldexpf(lo[3], s), h[2], l[2]);
                q4_split(ldexpf(hi[1], s), ldexpf(hi[3], s), h[3], l[3]);
                xh[tt] = as_f16x8(h[0], h[1], h[2], h[3]);
                xl[tt] = as_f16x8(l[0], l[1], l[2], l[3]);
            }
            // a row tile's sums join its accumulators under the next one's products
            f32x4 c[2][TT];
            auto fold = [&](int rt) {
                const f16x2 d2 = as_f16x2(ds[rt / 2][i]);
                const _Float16 d = rt % 2 ? d2.y : d2.x;
#pragma unroll
                for (int tt = 0; tt < TT; ++tt)
#pragma unroll
                    for (int r = 0; r < 4; ++r) acc[rt][tt][r] = fmaf((float)d, c[rt & 1][tt][r], acc[rt][tt][r]);
            };
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
                const f16x8 wf = q4_f16(nib[rt][i], km);
#pragma unroll
                for (int tt = 0; tt < TT; ++tt)
                    c[rt & 1][tt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xl[tt], wf, f32x4{0, 0, 0, 0}, 0, 0, 0);
#pragma unroll
                for (int tt = 0; tt < TT; ++tt)
                    c[rt & 1][tt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xh[tt], wf, c[rt & 1][tt], 0, 0, 0);
                if (rt > 0) fold(rt - 1);
                // the next loads a few at a time (past the part they read its last block again)
                if (rt < TT) load_x(b + PB, i % PB, rt);
                if (RT >= 4 ? rt >= RT - RT / 4 : i < RT && rt == RT - 1)
                    load_w(c0 + 4, RT >= 4 ? i * (RT / 4) + rt - (RT - RT / 4) : i);
                __builtin_amdgcn_sched_barrier(0);
            }
            fold(RT - 1);
        }
    }
    // the parts' sums meet in LDS; wave p finishes every fourth (row tile, token tile)
#pragma unroll
    for (int tt = 0; tt < TT; ++tt) {
        int sh[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) sh[r] = __shfl(E[tt], 4 * g + r) - 141;
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
            ps[p][rt][tt][lane] = make_float4(ldexpf(acc[rt][tt][0], sh[0]), ldexpf(acc[rt][tt][1], sh[1]),
                                              ldexpf(acc[rt][tt][2], sh[2]), ldexpf(acc[rt][tt][3], sh[3]));
    }
    __syncthreads();
    float *y = mat.y;
#pragma unroll
    for (int i = 0; i < (RT * TT + 3) / 4; ++i) {
        const int q = 4 * i + p, tt = q % TT, rt = q / TT;
        if (RT * TT % 4 != 0 && q >= RT * TT) break;
        const int t = t0 + 16 * tt + 4 * g, row = r0 + 16 * rt + j;
        const float4 a = ps[0][rt][tt][lane], b = ps[1][rt][tt][lane], c = ps[2][rt][tt][lane], d = ps[3][rt][tt][lane];
        const float o[4] = {(a.x + b.x) + (c.x + d.x), (a.y + b.y) + (c.y + d.y), (a.z + b.z) + (c.z + d.z),
                            (a.w + b.w) + (c.w + d.w)};
#pragma unroll
        for (int r = 0; r < 4; ++r)
            if (t + r < n_in && row < n_out) y[(size_t)(t + r) * n_out + row] = o[r];
    }
}

// ---- Many rows (a vocabulary head): exact int8 block sums on the matrix cores. The token's activations
// become, per block b, four int8 digits D_p (|D_p| <= 64) with
//   x_k 2^(132 - E_b) = D_0k + D_1k 2^-7 + D_2k 2^-14 + D_3k 2^-21 (+ less than 2^-22),
// E_b the largest biased exponent of the block's |x| (so |x_k| 2^(132 - E_b) < 64): exact for every
// element within 2^-3 of the block's largest, and within 2^-28 of that largest for the rest. Each
// v_mfma_i32_16x16x32_i8 then sums 16 (n - 8) D over one block's 8 elements exactly, with the
// weights 16 (n - 8) = ((n ^ 8) << 4) as signed bytes. A step covers 16 rows x 4 blocks: K group g of
// the instruction carries one block of each row (B, from lane (row j, group g)), and A row 4g + p
// carries digit p of that block (zero in the other groups), so lane (j, g) receives C[4g + p][j], the
// four digit sums of its own row and block, which it folds with its own d:
//   acc += d * (((128 C_2 + C_3) 2^-14 + (128 C_0 + C_1)) * 2^(E_b - 143)),
// the block's term d sum_k (n_k - 8) x_k up to f32 rounding. The lanes of a row add their sums in
// a fixed order, and the tokens of a pass (up to 4 per blockIdx.y) share only the weight loads, so
// a token's result does not depend on the other tokens of the call. A block with a non-finite
// activation gives NaN rows.
typedef int qi_v4i __attribute__((ext_vector_type(4)));

// Digits of four elements (p: digit, bytes: elements) for blocks whose largest exponent is e.
__device__ __forceinline__ void qi_digits(float4 v, int e, uint32_t (&pk)[4]) {
    const float e4[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int p = 0; p < 4; ++p) pk[p] = 0u;
#pragma unroll
    for (int el = 0; el < 4; ++el) {
        float u = ldexpf(e4[el], 132 - e);
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            const float dp = rintf(u);
            pk[p] |= ((uint32_t)(int)dp & 0xFFu) << (8 * el);
            u = (u - dp) * 128.0f;
        }
    }
}
// The largest biased exponent of a block, of which each of 8 lanes holds four elements.
__device__ __forceinline__ int qi_exponent(float4 v) {
    int e = max(max(exp_field(v.x), exp_field(v.y)), max(exp_field(v.z), exp_field(v.w)));
    e = max(e, __shfl_xor(e, 1));
    e = max(e, __shfl_xor(e, 2));
    return max(e, __shfl_xor(e, 4));
}
__device__ __forceinline__ float qi_scale(int e) { return e == 255 ? __uint_as_float(0x7FC00000u) : ldexpf(1.0f, e - 143); }
// 128 times the value of a block's four digit sums (|C_p| <= 2^18, so the pairs are exact in 32 bits)
__device__ __forceinline__ float qi_value(qi_v4i c) {
    return fmaf((float)(c[2] * 128 + c[3]), 6.103515625e-5f, (float)(c[0] * 128 + c[1]));
}
constexpr int QI_WAVES = 8, QI_ROWS = 16, QI_CH = 4;  // waves, rows per wave, step pairs per load chunk
constexpr int QI_BUF = 1;                               // chunks in registers
constexpr int QI_MIN_ROWS = 16384, QI_MAX_NB = 256;    // rvh_q4_mm takes this kernel from 16384 rows, k <= 8192
// dynamic LDS for tt tokens: digits [tt][nb][4 digits][8 dwords], 8 zero dwords, then the block
// scales [tt][nb]; passes take 4, 2 or 1 tokens, as many as fit 64 KB
inline size_t qi_lds_bytes(int nb, int tt) { return (size_t)tt * nb * (128 + 4) + 32; }
inline int qi_tokens(int nb, int n_in) {
    const int tt = qi_lds_bytes(nb, 4) <= 65536 ? 4 : (qi_lds_bytes(nb, 2) <= 65536 ? 2 : 1);
    return n_in >= tt ? tt : (n_in >= 2 && tt >= 2 ? 2 : 1);
}

// ALN: rows of an even block count on a 4-byte aligned matrix (q4_rows_aligned). TT: tokens per
// pass (blockIdx.y), which share the weight loads; each has its own digits, MFMAs and folds, the
// same operations as a pass of one token, so the same bits.
template <bool ALN, int TT>
__global__ __launch_bounds__(QI_WAVES * 64) void k_q4_mm_i8(const uint8_t *__restrict__ w, const float *__restrict__ x,
                                                  float *__restrict__ y, int n_out, int k, int n_in) {
    extern __shared__ __align__(16) uint32_t qi_sh[];
    const int nb = k / QK, tid = threadIdx.x;
    const int t0 = blockIdx.y * TT, nt = min(TT, n_in - t0);
    // token t's digits at dig + t nb 32, its block scales at xsc + t nb, one zero area after them
    uint32_t *dig = qi_sh, *zero = qi_sh + TT * nb * 32;
    float *xsc = (float *)(qi_sh + TT * nb * 32 + 8);
    const int lane = tid & 63, j = lane & 15, g = lane >> 4;
    const int r0 = (blockIdx.x * QI_WAVES + (tid >> 6)) * QI_ROWS;
    const size_t rb = (size_t)nb * Q4_BLOCK;
    const uint8_t *wr = w + (size_t)min(r0 + j, n_out - 1) * rb;
    // Steps go in pairs: K group g of pair p carries block 8p + 2g in the pair's first step and
    // block 8p + 2g + 1 in its second, so each lane loads two adjacent blocks, 36 bytes of its row.
    // This lane's A operand: digit j & 3 of its K group's block when j >> 2 == g, zeros otherwise.
    const bool adig = (j >> 2) == g;
    const int pairs = (nb + 7) >> 3, nch = (pairs + QI_CH - 1) / QI_CH;
    // a pair's weights: aligned rows, its 9 dwords as loaded (d0 in the low half of v[0], nibbles of
    // the first block from byte 2, d1 in the high half of v[4], nibbles of the second in v[5 .. 8]);
    // otherwise v = {d0, n0[4], d1, n1[4]}
    auto load = [&](int c, uint32_t (&v)[QI_CH][10]) {
#pragma unroll
        for (int u = 0; u < QI_CH; ++u) {
            const int b0 = (c * QI_CH + u) * 8 + 2 * g;
            if constexpr (ALN) {
                // blocks 2i and 2i + 1 are the 9 dwords from byte 36 i (rows of an even block count)
                const Dwords<4> a = *(const Dwords<4> *)(wr + min(b0, nb - 2) * Q4_BLOCK);
                const Dwords<4> e = *(const Dwords<4> *)(wr + min(b0, nb - 2) * Q4_BLOCK + 16);
                const uint32_t f = *(const uint32_t *)(wr + min(b0, nb - 2) * Q4_BLOCK + 32);
                // the dwords as loaded: compute() picks the fields, so nothing here waits for them
                const uint32_t dw[9] = {a.q[0], a.q[1], a.q[2], a.q[3], e.q[0], e.q[1], e.q[2], e.q[3], f};
#pragma unroll
                for (int i = 0; i < 9; ++i) v[u][i] = dw[i];
            } else {
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const uint8_t *p = wr + min(b0 + h, nb - 1) * Q4_BLOCK;
                    v[u][5 * h] = *(const uint16_t *)p;
                    const Q4Nibbles<4> q = *(const Q4Nibbles<4> *)(p + 2);
#pragma unroll
                    for (int m = 0; m < 4; ++m) v[u][5 * h + 1 + m] = q.q[m];
                }
            }
        }
    };
    // The token's activations first (a thread per 4 elements, 8 threads per block), then the first
    // QI_BUF chunks of weights, in flight while the activation digits are built; chunk c + QI_BUF is
    // loaded into chunk c's registers once chunk c is computed. (Loads past the last chunk would
    // re-read it; with more than one chunk in registers, skipping them under a branch makes the
    // compiler's waits on the other path wait for the newer loads too.)
    constexpr int XPT = QI_MAX_NB * 8 / (QI_WAVES * 64);  // float4s per thread and token at most
    float4 xq[TT][XPT];
#pragma unroll
    for (int t = 0; t < TT; ++t) {
        const float4 *xt = (const float4 *)(x + (size_t)(t0 + min(t, nt - 1)) * k);
#pragma unroll
        for (int i = 0; i < XPT; ++i) {
            const int f = tid + i * QI_WAVES * 64;
            xq[t][i] = f < nb * 8 ? xt[f] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        }
    }
    const bool rows_live = r0 < n_out;
    uint32_t vb[QI_BUF][QI_CH][10];
#pragma unroll
    for (int i = 0; i < QI_BUF; ++i)
        if (i < nch) load(i, vb[i]);
    // the digits
#pragma unroll
    for (int t = 0; t < TT; ++t)
#pragma unroll
    for (int i = 0; i < XPT; ++i) {
        const int f = tid + i * QI_WAVES * 64;
        if (t >= nt || f >= nb * 8) break;
        const int blk = t * nb + (f >> 3), q = f & 7;
        const float4 v = xq[t][i];
        const int e = qi_exponent(v);
        uint32_t pk[4];
        qi_digits(v, e, pk);
        // elements 4q .. 4q+3 are bytes 8q .. 8q+3 of a digit's 32 (q < 4); 16 + 4m .. are 8m+4 ..
        const int dw = q < 4 ? 2 * q : 2 * (q - 4) + 1;
#pragma unroll
        for (int p = 0; p < 4; ++p) dig[(blk * 4 + p) * 8 + dw] = pk[p];
        if (q == 0) xsc[blk] = qi_scale(e);
    }
    if (tid < 8) zero[tid] = 0u;
    __syncthreads();
    if (!rows_live) return;

    float acc[TT];
#pragma unroll
    for (int t = 0; t < TT; ++t) acc[t] = 0.0f;
    auto compute = [&](int c, const uint32_t (&v)[QI_CH][10]) {
#pragma unroll
        for (int u = 0; u < QI_CH; ++u) {
            if (c * QI_CH + u >= pairs) break;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int blk = (c * QI_CH + u) * 8 + 2 * g + h;
                const bool live = blk < nb;
                uint32_t nib[4], dbits;
                if constexpr (ALN) {
#pragma unroll
                    for (int m = 0; m < 4; ++m)
                        nib[m] = h ? v[u][5 + m] : __builtin_amdgcn_perm(v[u][m + 1], v[u][m], 0x05040302u);
                    dbits = h ? v[u][4] >> 16 : v[u][0] & 0xFFFFu;
                } else {
#pragma unroll
                    for (int m = 0; m < 4; ++m) nib[m] = v[u][5 * h + 1 + m];
                    dbits = v[u][5 * h];
                }
                long bw[4];
#pragma unroll
                for (int m = 0; m < 4; ++m) {
                    const uint32_t n8 = nib[m] ^ 0x88888888u;
                    bw[m] = (long)(((uint64_t)(n8 & 0xF0F0F0F0u) << 32) | ((n8 << 4) & 0xF0F0F0F0u));
                }
                const float dv = h2f((uint16_t)dbits);
#pragma unroll
                for (int tk = 0; tk < TT; ++tk) {
                    if (tk >= nt) break;
                    const uint32_t *ap = adig && live ? dig + ((tk * nb + blk) * 4 + (j & 3)) * 8 : zero;
                    const uint4 a0 = *(const uint4 *)ap, a1 = *(const uint4 *)(ap + 4);
                    const uint32_t ad[8] = {a0.x, a0.y, a0.z, a0.w, a1.x, a1.y, a1.z, a1.w};
                    qi_v4i cm = {0, 0, 0, 0};
#pragma unroll
                    for (int m = 0; m < 4; ++m) {
                        const long aw = (long)(((uint64_t)ad[2 * m + 1] << 32) | ad[2 * m]);
                        cm = __builtin_amdgcn_mfma_i32_16x16x32_i8(aw, bw[m], cm, 0, 0, 0);
                    }
                    const float t = qi_value(cm);
                    // past the row's last block the lane adds nothing (its loaded d is another block's)
                    if (live) acc[tk] = fmaf(dv, t * xsc[tk * nb + blk], acc[tk]);
                }
            }
        }
    };
    for (int c0 = 0; c0 < nch; c0 += QI_BUF) {
#pragma unroll
        for (int b = 0; b < QI_BUF; ++b) {
            const int c = c0 + b;
            if (c >= nch) break;
            compute(c, vb[b]);
            if (c + QI_BUF < nch) load(c + QI_BUF, vb[b]);
        }
    }
    // the four lanes of row j, groups (0 + 2) + (1 + 3)
#pragma unroll
    for (int t = 0; t < TT; ++t) {
        if (t >= nt) break;
        float r = acc[t] + __shfl_xor(acc[t], 32);
        r = r + __shfl_xor(r, 16);
        if (g == 0 && r0 + j < n_out) y[(size_t)(t0 + t) * n_out + r0 + j] = r;
    }
}

// The same sums for more tokens than k_q4_mm_i8 takes in a pass: 4 NQ tokens and 16 RT rows a wave. One
// MFMA covers one block of 16 rows and four tokens (A row 4t + p: digit p of token t; K group g: dword g
// of the block), so lane (j, g) receives the four digit sums of weight row j and token g: the integers of
// k_q4_mm_i8, whose four K groups' sums this lane keeps as four accumulators, adds in the same order and
// so with the same bits. Workgroups of 8 waves take 128 RT rows and share the digits of 8 blocks at a
// time in LDS, formed by the whole workgroup between the 8 before and these. What bounds it: VALU, 7
// instructions to fold a block's sums per row and token (64 rows and 32 tokens a wave: 262,144 x 2816 in
// 254 us, 1.63 TB/s of the matrix, 186 TFLOP/s; the folds alone are 137 us of VALU; digits that 16 lanes
// read from 512 bytes instead of 128 took 258, 20,000 x 2816 66 instead of 51).
constexpr int QH_CB = 8;  // blocks per chunk
template <int NQ, int RT, bool ALN>
__global__ __launch_bounds__(QI_WAVES * 64) void k_q4_i8_tile(const uint8_t *__restrict__ w, const float *__restrict__ x,
                                                              float *__restrict__ y, int n_out, int k, int n_in) {
    // [buffer][block][quad][K group][A row][half]: 16 lanes read 128 bytes in a row; a block's pitch is two
    // dwords past a multiple of the banks, for the stores of eight blocks at once
    constexpr int DP = NQ * 128 + 2;
    __shared__ __attribute__((aligned(16))) uint32_t dig[2][QH_CB * DP];
    __shared__ __attribute__((aligned(16))) float xsc[2][QH_CB][4][NQ];         // token 4 q + g at [g][q]
    constexpr int XP = NQ / 2;  // float4s of x per thread and chunk
    const int tid = threadIdx.x, lane = tid & 63, j = lane & 15, g = lane >> 4;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nb = k / QK, nch = (nb + QH_CB - 1) / QH_CB, t0 = blockIdx.y * 4 * NQ;
    const int r0 = (blockIdx.x * QI_WAVES + wv) * 16 * RT;
    const uint8_t *wr[RT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) wr[rt] = w + (size_t)min(r0 + 16 * rt + j, n_out - 1) * ((size_t)nb * Q4_BLOCK);
    uint32_t v[RT][10];
    auto load_w = [&](int c, int rt) {
        const int b = c * QH_CB + 2 * g;
        if constexpr (ALN) {
            const uint8_t *a = wr[rt] + min(b, nb - 2) * Q4_BLOCK;
            const Dwords<4> d0 = *(const Dwords<4> *)a, d1 = *(const Dwords<4> *)(a + 16);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                v[rt][i] = d0.q[i];
                v[rt][4 + i] = d1.q[i];
            }
            v[rt][8] = *(const uint32_t *)(a + 32);
        } else {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const uint8_t *a = wr[rt] + min(b + h, nb - 1) * Q4_BLOCK;
                const Q4Nibbles<4> q = *(const Q4Nibbles<4> *)(a + 2);
                v[rt][5 * h] = *(const uint16_t *)a;
#pragma unroll
                for (int i = 0; i < 4; ++i) v[rt][5 * h + 1 + i] = q.q[i];
            }
        }
    };
    // x of a chunk: wave wv takes token 8 i + wv in its pass i, lane l elements 4 (l % 8) .. of block l / 8
    float4 xv[XP];
    auto load_x = [&](int c) {
#pragma unroll
        for (int i = 0; i < XP; ++i) {
            const float *xt = x + (size_t)min(t0 + 8 * i + wv, n_in - 1) * k;
            xv[i] = buffer_load4(buffer_rsrc(xt, (uint32_t)nb * QK * 4), (uint32_t)(c * QH_CB * QK + 4 * lane) * 4, 0);
        }
    };
    auto digits = [&](int c) {
#pragma unroll
        for (int i = 0; i < XP; ++i) {
            const int t = 8 * i + wv, q = lane & 7, b = lane >> 3, e = qi_exponent(xv[i]);
            uint32_t pk[4];
            qi_digits(xv[i], e, pk);
#pragma unroll
            for (int p = 0; p < 4; ++p)
                dig[c & 1][b * DP + (t >> 2) * 128 + (q & 3) * 32 + (4 * (t & 3) + p) * 2 + (q >> 2)] = pk[p];
            if (q == 0) xsc[c & 1][b][t & 3][t >> 2] = qi_scale(e);
        }
    };
    load_x(0);
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) load_w(0, rt);
    float acc[RT][NQ][4];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int q = 0; q < NQ; ++q)
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[rt][q][i] = 0.0f;
    digits(0);
    __syncthreads();
    for (int c = 0; c < nch; ++c) {
        const bool more = c + 1 < nch;
        load_x(c + 1);  // past the row: zeros
        uint32_t nib[RT][2][4], ds[RT][4];
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            uint32_t s;
            if constexpr (ALN) {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    nib[rt][0][i] = __builtin_amdgcn_perm(v[rt][i + 1], v[rt][i], 0x05040302u);
                    nib[rt][1][i] = v[rt][5 + i];
                }
                s = __builtin_amdgcn_perm(v[rt][4], v[rt][0], 0x07060100u);
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    nib[rt][0][i] = v[rt][1 + i];
                    nib[rt][1][i] = v[rt][6 + i];
                }
                s = v[rt][0] | v[rt][5] << 16;
            }
            // a block past the row weighs nothing, whatever it holds (its digits are zeros)
            if (c * QH_CB + 2 * g >= nb) s &= 0xFFFF0000u;
            if (c * QH_CB + 2 * g + 1 >= nb) s &= 0x0000FFFFu;
            rows_transpose(nib[rt][0]);
            rows_transpose(nib[rt][1]);
            rows_gather(s, ds[rt]);
        }
        // steps of a row tile and QS token quads: a step's sums are folded under the next step's products
        constexpr int QS = NQ < 4 ? NQ : 4;
        qi_v4i cm[2][QS];
#pragma unroll
        for (int i = 0; i < QH_CB; ++i) {
            long a[NQ];
            float xs[NQ];
#pragma unroll
            for (int q = 0; q < NQ; ++q) {
                a[q] = *(const long *)&dig[c & 1][i * DP + q * 128 + g * 32 + j * 2];
                xs[q] = xsc[c & 1][i][g][q];
            }
            auto fold = [&](int st) {
                const int rt = st / (NQ / QS), q0 = st % (NQ / QS) * QS;
                const f16x2 d2 = as_f16x2(ds[rt][i >> 1]);
                const _Float16 d = i & 1 ? d2.y : d2.x;
#pragma unroll
                for (int q = 0; q < QS; ++q)
                    acc[rt][q0 + q][i >> 1] = fmaf((float)d, qi_value(cm[st & 1][q]) * xs[q0 + q], acc[rt][q0 + q][i >> 1]);
                // in this step, and not where the sums are next used
                if constexpr (QS == 4)
                    asm volatile("" : "+v"(acc[rt][q0][i >> 1]), "+v"(acc[rt][q0 + 1][i >> 1]),
                                 "+v"(acc[rt][q0 + 2][i >> 1]), "+v"(acc[rt][q0 + 3][i >> 1]));
                else
                    asm volatile("" : "+v"(acc[rt][q0][i >> 1]), "+v"(acc[rt][q0 + 1][i >> 1]));
            };
            long bw;
#pragma unroll
            for (int st = 0; st < RT * NQ / QS; ++st) {
                const int rt = st / (NQ / QS), q0 = st % (NQ / QS) * QS;
                if (q0 == 0) {
                    const uint32_t n8 = nib[rt][i & 1][i >> 1] ^ 0x88888888u;
                    bw = (long)(((uint64_t)(n8 & 0xF0F0F0F0u) << 32) | ((n8 << 4) & 0xF0F0F0F0u));
                }
#pragma unroll
                for (int q = 0; q < QS; ++q)
                    cm[st & 1][q] = __builtin_amdgcn_mfma_i32_16x16x32_i8(a[q0 + q], bw, qi_v4i{0, 0, 0, 0}, 0, 0, 0);
                if (st > 0) fold(st - 1);
                if (st == 0 && i >= 4 && i - 4 < RT) load_w(min(c + 1, nch - 1), i - 4);
                __builtin_amdgcn_sched_barrier(0);
            }
            fold(RT * NQ / QS - 1);
        }
        if (more) digits(c + 1);
        __syncthreads();
    }
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
            const int t = t0 + 4 * q + g, row = r0 + 16 * rt + j;
            const float (&u)[4] = acc[rt][q];
            if (t < n_in && row < n_out) y[(size_t)t * n_out + row] = (u[0] + u[2]) + (u[1] + u[3]);
        }
}

// The workgroups of 16 rt rows of every matrix, from mats.n_out.
inline long q4_starts(Q4Mats &mats, int rt) {
    long s = 0;
    for (int m = 0; m < mats.n; ++m) {
        mats.start[m] = (int)s;
        s += grid_blocks(mats.n_out[m], 16 * rt);
        if (s > 0x7fffffffL - 8) return -1;
    }
    mats.start[mats.n] = (int)s;
    return s;
}

// The matrices of fewer than QI_MIN_ROWS rows, in one launch.
int q4_run(Q4Mats &mats, const float *x, int k, int n_in) {
    if (mats.n == 0) return 0;
    long rows = 0;
    for (int m = 0; m < mats.n; ++m) rows += mats.n_out[m];
    bool dwords = true, shifted = k / QK > 1;
    for (int m = 0; m < mats.n; ++m) {
        dwords = dwords && q4_rows_aligned(mats.w[m], k / QK);
        shifted = shifted && ((uintptr_t)mats.w[m] & 3) == 0;
    }
    const int cus = device_cus();
    // Up to four tokens a pass, each its own conversion in the wave (5 tokens: 40 us a layer's seven products
    // against 43 here), and more passes while they are two workgroups a CU (one for few tokens on rows that are not
    // on dwords): a tile's parts are longer chains. 5 tokens, 1000 x 4096 14 us in a tile, 8 here (8 f32
    // products on the VALU), 33 tokens, 512 x 2816 17 / 9; 4096 x 2816, 5 tokens 9.1 / 8.7, 8 of 8192 rows
    // 9.7 / 13; 4096 x 2080, 5 tokens 8.5 / 9.4.
    const long vec_wgs = q4_starts(mats, 1), passes = grid_blocks(n_in, 4);
    RVM_CHECK(vec_wgs > 0);
    if (n_in <= 4 || vec_wgs * passes <= (dwords || n_in > 16 ? 2L : 1L) * cus) {
        auto go = [&](auto kern) {
            hipLaunchKernelGGL(kern, dim3((unsigned)vec_wgs, (unsigned)passes), dim3(64 * Q4_PARTS), 0, cur_stream(),
                               mats, x, k, n_in);
        };
        auto by_loads = [&](auto ntc, auto npc) {
            constexpr int NT = decltype(ntc)::value, NP = decltype(npc)::value;
            if (dwords) go(k_q4_vec<NT, NP, QV_DWORDS>);
            else if (shifted) go(k_q4_vec<NT, NP, QV_SHIFTED>);
            else go(k_q4_vec<NT, NP, QV_SPLIT>);
        };
        auto by_passes = [&](auto ntc) {
            switch (min(QV_CH, grid_blocks(q4_part(k / QK), 8))) {
                case 1: by_loads(ntc, std::integral_constant<int, 1>{}); break;
                case 2: by_loads(ntc, std::integral_constant<int, 2>{}); break;
                case 3: by_loads(ntc, std::integral_constant<int, 3>{}); break;
                default: by_loads(ntc, std::integral_constant<int, 4>{}); break;
            }
        };
        if (n_in == 1) by_passes(std::integral_constant<int, 1>{});
        else if (n_in == 2) by_passes(std::integral_constant<int, 2>{});
        else by_passes(std::integral_constant<int, 4>{});
        return launched();
    }
    // Then tiles of 16 tokens, or 32.
    const int tt = n_in > 16 ? 2 : 1, ty = grid_blocks(n_in, 16 * tt);
    RVM_CHECK(ty <= 65535);
    // The largest tile of which there are still 35/64 of the CUs (140 of 256): a larger tile converts each x
    // and each nibble for more products, which outweighs idle CUs until about there. One layer's seven
    // projections, at least 512 / 220 / 140 / 110 workgroups: 250 tokens 189 / 168 / 152 / 152 us, 100
    // tokens 137 / 122 / 100 / 99, 16 tokens 47.7 / 47.7 / 47.8 / 50.8; 500 tokens at width 1024 123 / 104 /
    // 104 / 117.
    int rt = 8;
    while (rt > 2 && (rows + 16 * rt - 1) / (16 * rt) * ty < 35L * cus / 64) rt >>= 1;
    const long wgs = q4_starts(mats, rt);
    RVM_CHECK(wgs > 0);
    auto go = [&](auto kern) {
        hipLaunchKernelGGL(kern, dim3((unsigned)((wgs + 7) / 8 * 8), ty), dim3(256), 0, cur_stream(), mats, x, k, n_in);
    };
    if (tt == 2) rt == 8 ? go(k_q4_tile<8, 2, 1>) : rt == 4 ? go(k_q4_tile<4, 2, 2>) : go(k_q4_tile<2, 2, 4>);
    else rt == 8 ? go(k_q4_tile<8, 1, 4>) : rt == 4 ? go(k_q4_tile<4, 1, 4>) : go(k_q4_tile<2, 1, 4>);
    return launched();
}

// a matrix of n_out rows of k goes through k_q4_mm_i8 (whatever the token count)
inline bool q4_uses_i8(int n_out, int k) { return n_out >= QI_MIN_ROWS && k / QK <= QI_MAX_NB; }

int q4_run_i8(const uint8_t *w, const float *x, float *y, int n_out, int k, int n_in) {
    const int nb = k / QK;
    const bool aln = q4_rows_aligned(w, nb);
    // From 5 tokens (3 on rows that are not on dwords) 8, 16 or 32 a pass over the matrix: 262,144 x 2816, 32
    // tokens 254 us (eight passes of 4 tokens 897), 8 tokens 120 (228); 100,000 x 2080 unaligned, 4 tokens:
    // 67 in a pass of 4, 57 here; 40,001 x 4096, 4 tokens: 42 in a pass of 4, 47 here. Two tokens a pass (where
    // four tokens' digits do not fit 64 KB) still win while all passes are two workgroups a CU: 16,384 x 4096,
    // 5 tokens 27 / 32, 8 tokens 29 / 32; 20,000 rows 30 / 33 and 44 / 33.
    const int cus = device_cus(), tt = qi_tokens(nb, n_in), tiles = grid_blocks(n_out, QI_WAVES * 16);
    if (n_in > (aln ? 4 : 2) && !(aln && tt == 2 && (long)tiles * grid_blocks(n_in, 2) <= 2L * cus)) {
        // Half the tokens a pass while the CUs take both passes at once: 16,384 x 2816, 9 tokens 28 us in a pass
        // of 16, 20 in two of 8; 32 tokens 52 in a pass of 32, 28 in two of 16. Then 16 rows a wave while
        // those workgroups fit the CUs, and 32 (64 for 32 tokens) as long: the more rows a workgroup shares its digits
        // with the longer it takes, 52 / 75 / 122 us a round at 32 tokens and k 2816 (32,768 rows 52 / 76 / 123;
        // 65,536 83 / 77 / 124; 100,000 154 / 149 / 124).
        int nq = n_in <= 8 ? 2 : n_in <= 16 ? 4 : 8;
        while (nq > 2 && (long)tiles * grid_blocks(n_in, 2 * nq) <= cus) nq >>= 1;
        const int rt = tiles <= cus ? 1 : nq == 8 && tiles > 2 * cus ? 4 : 2;
        RVM_CHECK(grid_blocks(n_in, 4 * nq) <= 65535);
        const dim3 grid(grid_blocks(n_out, QI_WAVES * 16 * rt), grid_blocks(n_in, 4 * nq));
        auto go = [&](auto kern) {
            hipLaunchKernelGGL(kern, grid, dim3(QI_WAVES * 64), 0, cur_stream(), w, x, y, n_out, k, n_in);
        };
        auto by_rows = [&](auto nqc) {
            constexpr int NQ = decltype(nqc)::value;
            if constexpr (NQ == 8) {
                if (rt == 4) {
                    aln ? go(k_q4_i8_tile<NQ, 4, true>) : go(k_q4_i8_tile<NQ, 4, false>);
                    return;
                }
            }
            if (rt == 2) aln ? go(k_q4_i8_tile<NQ, 2, true>) : go(k_q4_i8_tile<NQ, 2, false>);
            else aln ? go(k_q4_i8_tile<NQ, 1, true>) : go(k_q4_i8_tile<NQ, 1, false>);
        };
        if (nq == 2) by_rows(std::integral_constant<int, 2>{});
        else if (nq == 4) by_rows(std::integral_constant<int, 4>{});
        else by_rows(std::integral_constant<int, 8>{});
        return launched();
    }
    const dim3 grid(grid_blocks(n_out, QI_WAVES * QI_ROWS), grid_blocks(n_in, tt));
    auto go = [&](auto kern) {
        hipLaunchKernelGGL(kern, grid, dim3(QI_WAVES * 64), qi_lds_bytes(nb, tt), cur_stream(), w, x, y, n_out, k, n_in);
    };
    if (tt == 4) go(k_q4_mm_i8<true, 4>);
    else if (tt == 2) aln ? go(k_q4_mm_i8<true, 2>) : go(k_q4_mm_i8<false, 2>);
    else aln ? go(k_q4_mm_i8<true, 1>) : go(k_q4_mm_i8<false, 1>);
    return launched();
}

}  // namespace rvm

using namespace rvm;

extern "C" {

int rvh_q4_mm(const void *w, const float *x, float *y, int n_out, int k, int n_in) {
    const void *const ws[1] = {w};
    float *const ys[1] = {y};
    return rvm_q4_mm_n(1, ws, &n_out, ys, x, k, n_in);
}

int rvm_q4_mm_n(int n_mat, const void *const *w, const int *n_out, float *const *y, const float *x, int k, int n_in) {
    RVM_CHECK(n_mat >= 1 && n_mat <= Q4_NMAT && w && n_out && y && x && n_in > 0 && k > 0 && k % QK == 0);
    for (int m = 0; m < n_mat; ++m) RVM_CHECK(w[m] && y[m] && n_out[m] > 0 && ((uintptr_t)w[m] & 1) == 0);
    // a matrix's rows and width pick its arithmetic, whatever the token count
    Q4Mats mats{};
    for (int m = 0; m < n_mat; ++m) {
        if (q4_uses_i8(n_out[m], k)) {
            if (const int rc = q4_run_i8((const uint8_t *)w[m], x, y[m], n_out[m], k, n_in)) return rc;
            continue;
        }
        mats.w[mats.n] = (const uint8_t *)w[m];
        mats.y[mats.n] = y[m];
        mats.n_out[mats.n] = n_out[m];
        ++mats.n;
    }
    return q4_run(mats, x, k, n_in);
}

// The reference's K2 variant (rvhip.h:46-48) has rvh_q4_mm's result up to summation order and asks
// for 16-byte aligned x and 2-byte aligned w; here it is the same kernel.
int rvh_q4_mv(const void *w, const float *x, float *y, int n_out, int k, int n_in) {
    RVM_CHECK(((uintptr_t)x & 15) == 0);
    return rvh_q4_mm(w, x, y, n_out, k, n_in);
}

}  // extern "C"
