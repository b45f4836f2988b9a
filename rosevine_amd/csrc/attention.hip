// attention.hip - decode attention over a Q8_0 key/value ring with the reference's operator ABI
// (runtime/hip/rvhip.h:55-67): rvh_kv_store, rvh_attention, rvh_attn_split, rvh_attn_combine.
// The reference's kernels are runtime/hip/rvhip.hip:214-394, its host side runtime/src/hip.rs:423-530.
//
// Semantics (the reference's): query t of a call sits at position pos = p0 + t and attends, with
// scale 1.0, to keys lo .. pos, lo = max(0, pos + 1 - window) when window > 0, else 0. Key p is ring
// slot p % cap: row (slot * n_kv + g) of hd/32 Q8_0 blocks, g = h / (n_head / n_kv). Split-K cuts a
// query's keys into n_chunks contiguous chunks of ceil(len / n_chunks) keys; with more than one
// chunk each (query head, chunk) leaves an unnormalised partial {max, sum, acc[hd]} that
// rvh_attn_combine merges. Results match the CPU ops (runtime/tests/hip_ops.rs:245-271) to the
// reference's relative L2 bound of 1e-5; only summation orders differ.
//
// Work layout. A workgroup of 4 waves takes one tile (token, kv head, chunk) and G query heads that
// share the kv head (G up to the heads per kv head: fewer when the call has few tiles, to spread
// them over more CUs; the head groups of one tile run on one XCD). Keys go in tiles of 64:
//  - loads: wave w reads keys 16 w .. 16 w + 15 of the tile, key and value rows whole and
//    coalesced (lane l the quants of its DPL dimensions); the key quants go through LDS.
//  - scores: MFMA, heads x keys over one Q8_0 block (see k_attn_split); wave w takes the blocks
//    w, w + 4, ... of every key, and the four partial scores meet in LDS.
//  - softmax: wave w keeps its own online softmax over its 16 keys, the maxima and sums running
//    over the 16 lanes of a row.
//  - values: wave w accumulates its 16 keys into every dimension of every head (lane l owns
//    dimensions DPL l .. DPL l + DPL - 1), each key's weight read from the lane that scored it.
//  - merge: the four waves' (max, sum, values) combine in LDS after one barrier.
// Every workgroup is a short serial chain of loads; the grid fits the GPU in one round.
#include "internal.hpp"

namespace rvm {

constexpr int AT_WAVES = 4;
constexpr int AT_TILE = 64;    // keys per tile
constexpr int AT_MAXHD = 512;  // dimensions per head (8 per lane)

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef int v2i_t __attribute__((ext_vector_type(2)));

struct __attribute__((packed, aligned(2))) Q8Half {  // 8 quants of a Q8_0 block
    uint32_t q[2];
};
struct __attribute__((packed, aligned(2))) Q8Word {
    uint32_t q;
};

__device__ __forceinline__ float readlane_f(float v, int l) {
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), l));
}

// Max over the wave (NaN ignored), the same in every lane.
__device__ __forceinline__ float wave_max_f(float m) {
    m = half_max(m);
    return fmaxf(readlane_f(m, 0), readlane_f(m, 32));
}

__device__ __forceinline__ float q8_at(uint32_t u, int e) { return (float)(int8_t)(uint8_t)(u >> (8 * e)); }

// Max and sum over each row of 16 lanes (xor-pattern exchanges, so that every lane of the row ends
// with the same bits).
__device__ __forceinline__ float row16_max_f(float v) {
    v = maxf_bits(v, dpp<0xb1>(__builtin_bit_cast(uint32_t, v)));
    v = maxf_bits(v, dpp<0x4e>(__builtin_bit_cast(uint32_t, v)));
    v = maxf_bits(v, dpp<0x141>(__builtin_bit_cast(uint32_t, v)));
    return maxf_bits(v, dpp<0x140>(__builtin_bit_cast(uint32_t, v)));
}
__device__ __forceinline__ float row16_sum_f(float v) {
    v += __builtin_bit_cast(float, dpp<0xb1>(__builtin_bit_cast(uint32_t, v)));
    v += __builtin_bit_cast(float, dpp<0x4e>(__builtin_bit_cast(uint32_t, v)));
    v += __builtin_bit_cast(float, dpp<0x141>(__builtin_bit_cast(uint32_t, v)));
    return v + __builtin_bit_cast(float, dpp<0x140>(__builtin_bit_cast(uint32_t, v)));
}

// Four int8 quants as bf16 pairs (exact: |q| <= 128 has at most 8 significant bits): the f32
// value's high half is its bf16.
__device__ __forceinline__ void q8_bf16(uint32_t u, uint32_t &lo, uint32_t &hi) {
    const uint32_t f0 = __builtin_bit_cast(uint32_t, q8_at(u, 0)), f1 = __builtin_bit_cast(uint32_t, q8_at(u, 1));
    const uint32_t f2 = __builtin_bit_cast(uint32_t, q8_at(u, 2)), f3 = __builtin_bit_cast(uint32_t, q8_at(u, 3));
    lo = __builtin_amdgcn_perm(f1, f0, 0x07060302u);
    hi = __builtin_amdgcn_perm(f3, f2, 0x07060302u);
}

template <int DPL>
struct AttnTile {              // the wave's 16 keys of a tile, as loaded: row by row, coalesced
    uint32_t kq[16][DPL / 4];  // key rows: the lane's DPL quants (dimensions DPL l ..)
    uint16_t kd[16];           // and their block scale
    uint32_t vq[16][DPL / 4];  // value rows, likewise
    uint16_t vd[16];
};

// G query heads per workgroup; DPL contiguous value dimensions per lane (4 for hd <= 256, 8 for
// hd <= 512): lane l owns dimensions DPL l .. DPL l + DPL - 1, inside one Q8_0 block.
//
// Rows are read whole and coalesced (wave w reads keys 16 w .. 16 w + 15 of a tile, lane l the
// quants of its dimensions); the key quants then go through LDS into the MFMA layout.
//
// Scores run on v_mfma_f32_16x16x32_bf16 with the heads as rows (A = q), the keys as columns
// (B = key quants) and one Q8_0 block as the 32-long reduction: q is held exactly as the sum of
// three bf16 parts (8 + 8 + 8 significant bits), each a separate product accumulated in f32, and
// int8 quants are exact in bf16, so a block's partial is the f32 sum of exact products; the
// lane then scales its own key's partial by the block scale. Wave w takes blocks w, w + 4, ... of
// every key in the tile; lane l of the MFMA output holds heads 4 (l / 16) .. + 3 of key l % 16.
template <int G, int DPL>
__global__ __launch_bounds__(AT_WAVES * 64) void k_attn_split(
    const float *__restrict__ q, const uint8_t *__restrict__ kc, const uint8_t *__restrict__ vc,
    float *__restrict__ out, float *__restrict__ part, int n_tok, int n_head, int n_kv, int hd, int p0, int cap,
    int window, int n_chunks) {
    constexpr int NBW = DPL / 2;
    // LDS: partial scores [2][wave][key][head]; the tile's key quants [key][KROW bytes] and block
    // scales [key][16], whose space the waves' value sums [wave][head][dimension][lane] reuse
    constexpr int KROW = 64 * DPL + 16;  // padded: the 16 keys of a fragment read hit distinct banks
    constexpr int KBYTES = AT_TILE * KROW + AT_TILE * 16 * 2;
    constexpr int MBYTES = AT_WAVES * G * DPL * 64 * 4;
    __shared__ float red_lds[2 * AT_WAVES * AT_TILE * G];
    __shared__ __attribute__((aligned(16))) uint8_t kt_lds[KBYTES > MBYTES ? KBYTES : MBYTES];
    uint8_t *const kt_q = kt_lds;
    uint16_t *const kt_d = (uint16_t *)(kt_lds + AT_TILE * KROW);
    const int lane = threadIdx.x & 63, lr = lane & 15, lg = lane >> 4;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // workgroup -> (tile, head group): a tile is (token t, kv head g, chunk c); its S head groups
    // get workgroup numbers equal mod 8, so that they run on one XCD and share its L2 for the
    // tile's key and value rows
    const int S = (n_head / n_kv) / G;
    const int xcd = blockIdx.x & 7, rest = blockIdx.x >> 3;
    const int sg = rest % S;
    const long T = (long)(rest / S) * 8 + xcd;
    if (T >= (long)n_tok * n_kv * n_chunks) return;
    const int c = (int)(T % n_chunks);
    const int tg = (int)(T / n_chunks);
    const int g = tg % n_kv, t = tg / n_kv;
    const int h0 = g * (n_head / n_kv) + sg * G;
    const int pos = p0 + t;
    const int lo = window > 0 ? max(0, pos + 1 - window) : 0;
    const int len = pos - lo + 1;
    const int per = (len + n_chunks - 1) / n_chunks;
    const int k0 = lo + c * per, k1 = min(pos + 1, k0 + per);  // this chunk's keys [k0, k1)
    const int nb = hd / QK, row = nb * Q8_BLOCK;
    const size_t slot_bytes = (size_t)n_kv * row;
    const uint8_t *kg = kc + (size_t)g * row, *vg = vc + (size_t)g * row;

    // this lane's value dimensions DPL lane .. + DPL - 1, when below hd (hd is a multiple of 32)
    const bool vok = DPL * lane < hd;
    const int vd0 = vok ? DPL * lane : 0;
    const int vblk = (vd0 / QK) * Q8_BLOCK, vq_off = vblk + 2 + vd0 % QK;

    // ---- every first load at once: the q fragments (q[head lr][block b, elements 8 lg .. + 7]),
    // then the first tile's key and value rows. Loads are unconditional (clamped addresses, the
    // values selected afterwards) so that each wait counts only what it needs.
    float qx[NBW][8];
#pragma unroll
    for (int i = 0; i < NBW; ++i) {
        const int b = w + AT_WAVES * i;
        const bool qok = b < nb && lr < G;
        const float *qr = q + ((size_t)t * n_head + h0 + (qok ? lr : 0)) * hd + (qok ? b : 0) * QK + 8 * lg;
#pragma unroll
        for (int e = 0; e < 8; ++e) qx[i][e] = qr[e];
    }
    AttnTile<DPL> tl;
    const int j0 = 16 * w;  // the wave's keys in the value phase
    // the tile at `base` (ring slot `bslot`; later slots follow by increments, no division per key):
    // the wave's 16 keys, key and value rows; keys past the chunk read the tile's first key
    auto row_offsets = [&](int base, int bslot, size_t *off) {
#pragma unroll
        for (int jj = 0; jj < 16; ++jj) {
            int s = bslot + j0 + jj;
            s = s >= cap ? s - cap : s;
            off[jj] = (size_t)(base + j0 + jj < k1 ? s : bslot) * slot_bytes;
        }
    };
    auto load_keys = [&](int base, int bslot) {
        size_t off[16];
        row_offsets(base, bslot, off);
#pragma unroll
        for (int jj = 0; jj < 16; ++jj) {
            const uint8_t *kr = kg + off[jj];
            tl.kd[jj] = *(const uint16_t *)(kr + vblk);
            if constexpr (DPL == 8) {
                const Q8Half k8 = *(const Q8Half *)(kr + vq_off);
                tl.kq[jj][0] = k8.q[0];
                tl.kq[jj][1] = k8.q[1];
            } else {
                tl.kq[jj][0] = ((const Q8Word *)(kr + vq_off))->q;
            }
        }
    };
    auto load_values = [&](int base, int bslot) {
        size_t off[16];
        row_offsets(base, bslot, off);
#pragma unroll
        for (int jj = 0; jj < 16; ++jj) {
            const uint8_t *vr = vg + off[jj];
            tl.vd[jj] = *(const uint16_t *)(vr + vblk);
            if constexpr (DPL == 8) {
                const Q8Half v8 = *(const Q8Half *)(vr + vq_off);
                tl.vq[jj][0] = v8.q[0];
                tl.vq[jj][1] = v8.q[1];
            } else {
                tl.vq[jj][0] = ((const Q8Word *)(vr + vq_off))->q;
            }
        }
    };
    // order: q and the first keys, then (once q is in) the first values; a wave holds at most 63
    // loads in flight, and the q conversion must not wait behind the value rows
    const int slot0 = k0 % cap;
    load_keys(k0, slot0);  // an empty chunk reads slot0 and uses nothing
    __builtin_amdgcn_sched_barrier(0);

    // ---- q as three bf16 parts (A fragments; heads past G and blocks past hd are zero)
    bf16x8 qa[NBW][3];
#pragma unroll
    for (int i = 0; i < NBW; ++i) {
        const bool qok = w + AT_WAVES * i < nb && lr < G;
        uint32_t pk[3][4];
#pragma unroll
        for (int e = 0; e < 8; e += 2) {
            f32x2 r = {qok ? qx[i][e] : 0.0f, qok ? qx[i][e + 1] : 0.0f};
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                const bf16x2 b = __builtin_convertvector(r, bf16x2);
                pk[k][e / 2] = __builtin_bit_cast(uint32_t, b);
                r -= __builtin_convertvector(b, f32x2);  // exact: the rounding's residual
            }
        }
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            uint4 v = {pk[k][0], pk[k][1], pk[k][2], pk[k][3]};
            qa[i][k] = __builtin_bit_cast(bf16x8, v);
        }
    }
    __builtin_amdgcn_sched_barrier(0);
    load_values(k0, slot0);

    // softmax statistics: each wave keeps its own over its keys; lane (j, r) = (lane % 16,
    // lane / 16) holds heads r HPL .. r HPL + HPL - 1 (rows r < RU)
    constexpr int HPL = G >= 4 ? G / 4 : 1, RU = G >= 4 ? 4 : G;
    float m[HPL], l[HPL], acc[G][DPL];
#pragma unroll
    for (int u = 0; u < HPL; ++u) {
        m[u] = -INFINITY;
        l[u] = 0.0f;
    }
#pragma unroll
    for (int h = 0; h < G; ++h)
#pragma unroll
        for (int e = 0; e < DPL; ++e) acc[h][e] = 0.0f;

    int buf = 0;
    for (int base = k0, bslot = slot0; base < k1;) {
        // ---- the wave's key rows into LDS (dimensions past hd are never read)
#pragma unroll
        for (int jj = 0; jj < 16; ++jj) {
            uint8_t *dst = kt_q + (j0 + jj) * KROW + DPL * lane;
            if constexpr (DPL == 8)
                *(uint2 *)dst = uint2{tl.kq[jj][0], tl.kq[jj][1]};
            else
                *(uint32_t *)dst = tl.kq[jj][0];
            if ((DPL * lane) % QK == 0) kt_d[(j0 + jj) * 16 + DPL * lane / QK] = tl.kd[jj];
        }
        __syncthreads();

        // ---- scores on MFMA: s[kg][r] = head 4 lg + r, key 16 kg + lr, over the wave's blocks
        f32x4 s[4];
#pragma unroll
        for (int kgp = 0; kgp < 4; ++kgp) s[kgp] = f32x4{0, 0, 0, 0};
#pragma unroll
        for (int i = 0; i < NBW; ++i) {
            const int b = w + AT_WAVES * i;
            if (b >= nb) break;
#pragma unroll
            for (int kgp = 0; kgp < 4; ++kgp) {
                const uint2 kw = *(const uint2 *)(kt_q + (16 * kgp + lr) * KROW + QK * b + 8 * lg);
                uint32_t kb[4];
                q8_bf16(kw.x, kb[0], kb[1]);
                q8_bf16(kw.y, kb[2], kb[3]);
                const bf16x8 bk = __builtin_bit_cast(bf16x8, uint4{kb[0], kb[1], kb[2], kb[3]});
                f32x4 d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(qa[i][0], bk, f32x4{0, 0, 0, 0}, 0, 0, 0);
                d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(qa[i][1], bk, d, 0, 0, 0);
                d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(qa[i][2], bk, d, 0, 0, 0);
                const float dk = h2f(kt_d[(16 * kgp + lr) * 16 + b]);
#pragma unroll
                for (int r = 0; r < 4; ++r) s[kgp][r] = fmaf(dk, d[r], s[kgp][r]);
            }
        }
        float *red = red_lds + buf * (AT_WAVES * AT_TILE * G);
#pragma unroll
        for (int kgp = 0; kgp < 4; ++kgp)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (4 * lg + r < G) red[(w * AT_TILE + 16 * kgp + lr) * G + 4 * lg + r] = s[kgp][r];
        __syncthreads();

        // ---- online softmax of the wave's keys 16 w .. 16 w + 15: lane (j, r) scores key 16 w + j
        // for its heads; maxima and sums run over the 16 lanes of each row
        const bool live = base + j0 + lr < k1;
        float p[HPL], corr[HPL];
#pragma unroll
        for (int u = 0; u < HPL; ++u) {
            const int h = (lg < RU ? lg : 0) * HPL + u;
            const int kk = j0 + lr;
            const float sc = ((red[kk * G + h] + red[(AT_TILE + kk) * G + h]) + red[(2 * AT_TILE + kk) * G + h]) +
                             red[(3 * AT_TILE + kk) * G + h];
            const float mn = fmaxf(m[u], row16_max_f(live ? sc : -INFINITY));
            corr[u] = m[u] == -INFINITY ? 0.0f : expf(m[u] - mn);
            p[u] = live ? expf(sc - mn) : 0.0f;
            l[u] = l[u] * corr[u] + row16_sum_f(p[u]);
            m[u] = mn;
        }

        // ---- values: the wave's 16 keys; dead keys weigh 0
        if (base + j0 < k1) {
#pragma unroll
            for (int h = 0; h < G; ++h) {
                const float ch = readlane_f(corr[h % HPL], 16 * (h / HPL));
#pragma unroll
                for (int e = 0; e < DPL; ++e) acc[h][e] *= ch;
            }
#pragma unroll
            for (int jj = 0; jj < 16; ++jj) {
                float x[DPL];
                const float d = h2f(tl.vd[jj]);
#pragma unroll
                for (int e = 0; e < DPL; ++e) x[e] = d * q8_at(tl.vq[jj][e / 4], e % 4);
#pragma unroll
                for (int h = 0; h < G; ++h) {
                    const float ph = readlane_f(p[h % HPL], 16 * (h / HPL) + jj);
#pragma unroll
                    for (int e = 0; e < DPL; ++e) acc[h][e] = fmaf(ph, x[e], acc[h][e]);
                }
            }
        }

        // ---- the next tile's rows, when there is one (issued last, so that no wait above counts them)
        const int next = base + AT_TILE;
        int nslot = bslot + AT_TILE;
        while (nslot >= cap) nslot -= cap;
        if (next < k1) {
            load_keys(next, nslot);
            load_values(next, nslot);
        }
        buf ^= 1;
        base = next;
        bslot = nslot;
    }

    // ---- merge the four waves: M = max of their maxima, their sums weighted by e^(m_w - M) and
    // added in wave order; one barrier, then each wave finishes a share of the (head, 4 dimensions)
    // groups. The value sums reuse the key tile's LDS, which the last tile's barrier has released.
    __shared__ float wm[AT_WAVES][G], wl[AT_WAVES][G];
    float *mrg = (float *)kt_lds;  // [wave][head * DPL + e][lane]
    __syncthreads();  // every wave is done with the last key tile
    if (lr == 0 && lg < RU)
#pragma unroll
        for (int u = 0; u < HPL; ++u) {
            wm[w][lg * HPL + u] = m[u];
            wl[w][lg * HPL + u] = l[u];
        }
#pragma unroll
    for (int h = 0; h < G; ++h)
#pragma unroll
        for (int e = 0; e < DPL; ++e) mrg[((size_t)w * G * DPL + h * DPL + e) * 64 + lane] = acc[h][e];
    __syncthreads();
    const size_t r0 = (size_t)t * n_head + h0;
    constexpr int NQ = G * DPL / 4;  // (head, 4 dimensions) groups
#pragma unroll
    for (int g0 = 0; g0 < NQ; g0 += AT_WAVES) {
        const int gi = g0 + w;
        if (NQ % AT_WAVES != 0 && gi >= NQ) break;
        const int h = gi / (DPL / 4), e0 = 4 * (gi % (DPL / 4));
        const float Mh = fmaxf(fmaxf(wm[0][h], wm[1][h]), fmaxf(wm[2][h], wm[3][h]));
        float f[AT_WAVES], den = 0.0f;
#pragma unroll
        for (int u = 0; u < AT_WAVES; ++u) {
            f[u] = wm[u][h] == -INFINITY ? 0.0f : expf(wm[u][h] - Mh);
            den = fmaf(f[u], wl[u][h], den);
        }
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            float num = 0.0f;
#pragma unroll
            for (int u = 0; u < AT_WAVES; ++u) num = fmaf(f[u], mrg[((size_t)u * G * DPL + h * DPL + e0 + e) * 64 + lane], num);
            v[e] = num;
        }
        if (n_chunks == 1) {
            const float inv = 1.0f / den;
            if (vok)
#pragma unroll
                for (int e = 0; e < 4; ++e) out[(r0 + h) * hd + vd0 + e0 + e] = v[e] * inv;
        } else {
            float *pp = part + ((r0 + h) * n_chunks + c) * (size_t)(hd + 2);
            if (e0 == 0 && lane == 0) {
                pp[0] = Mh;
                pp[1] = den;
            }
            if (vok)
#pragma unroll
                for (int e = 0; e < 4; ++e) pp[2 + vd0 + e0 + e] = v[e];
        }
    }
}

// ---- Streaming split-K for head dimensions 256 and 512 (nb = 8 or 16 Q8_0 blocks per row) ----
// A workgroup of 8 waves takes one tile (token, kv head, chunk) with up to 16 query heads of that kv
// head, so that every key and value row of the tile is read once. The tile's keys go in stages of
// 32, copied from HBM straight into LDS (global_load_lds, 1 KB of two or four whole rows per
// instruction) through a ring of ST_RING stages: ST_RING - 1 stages are in flight while one is
// computed, and each wave waits (vmcnt) only for the copies of the stage it needs next. A stage
// sits in LDS as [K/V][key][16-byte piece p ^ key] (piece p holds half of block p / 2's quants, read
// from the ring rows at 2-byte alignment; the XOR puts the same piece of 16 keys on distinct banks)
// and the block scales as the dwords that start at them (low half), [K/V][key][block].
//  - scores: v_mfma_f32_16x16x32_bf16, heads x 16 keys over one block (q as three exact bf16 parts,
//    the key quants exact in bf16), scaled by the key's block scale; wave w takes key group w & 1
//    and a quarter of the blocks, and the four partial scores meet in LDS;
//  - softmax: wave w keeps heads 2 w and 2 w + 1 (lane = head parity, key): their running max and
//    sum, and writes the stage's p and the rescale factor to LDS;
//  - values: v_mfma_f32_16x16x32_bf16 with A = p * d_v (heads x 32 keys, three exact bf16 parts)
//    and B = the value quants of 32 keys x 16 dimensions, read transposed out of LDS
//    (ds_read_b64_tr_b8: each 16-lane group turns 8 keys x 8 bytes into 8 dimensions x 8 keys);
//    wave w owns the dimensions of blocks w, w + 8, so no merge is needed.
constexpr int ST_WAVES = 8;
constexpr int ST_KEYS = 32;  // keys per stage
constexpr int ST_RING = 4;   // stages resident in LDS
constexpr int ST_PP = 36;    // row pitch of the p rows in LDS (floats)

template <int NB>
struct StreamShape {
    static constexpr int HD = 32 * NB;
    static constexpr int ROW = NB * Q8_BLOCK;
    static constexpr int QBYTES = 2 * ST_KEYS * HD;      // quants of a stage, K then V
    static constexpr int SBYTES = 2 * NB * ST_KEYS * 4;  // scale dwords of a stage
    static constexpr int STAGE = QBYTES + SBYTES;
    static constexpr int NQ = NB / 4;  // 16-byte copies per wave and stage
    static constexpr int NS = NB / 8;  // 4-byte copies per wave and stage
    static constexpr int NI = NQ + NS;
    static constexpr int SBW = NB / 4;  // blocks per wave in the scores
    static constexpr int VBW = NB / 8;  // blocks per wave in the values
    static constexpr int LDS = ST_RING * STAGE + (4 * 16 * ST_KEYS + 16 * ST_PP + 2 * 16) * 4;
    static_assert(LDS <= 163840, "LDS");
};

typedef __attribute__((address_space(3))) v2i_t lds_v2i_t;


__device__ __forceinline__ bf16x8 q8x8_bf16(uint32_t a, uint32_t b) {
    uint32_t k[4];
    q8_bf16(a, k[0], k[1]);
    q8_bf16(b, k[2], k[3]);
    return __builtin_bit_cast(bf16x8, uint4{k[0], k[1], k[2], k[3]});
}

// x as three bf16 parts whose sum is x exactly (each part the rounding of the residual before it)
__device__ __forceinline__ void split3_bf16(const float (&x)[8], bf16x8 (&a)[3]) {
    uint32_t pk[3][4];
#pragma unroll
    for (int e = 0; e < 8; e += 2) {
        f32x2 r = {x[e], x[e + 1]};
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const bf16x2 b = __builtin_convertvector(r, bf16x2);
            pk[k][e / 2] = __builtin_bit_cast(uint32_t, b);
            r -= __builtin_convertvector(b, f32x2);
        }
    }
#pragma unroll
    for (int k = 0; k < 3; ++k) a[k] = __builtin_bit_cast(bf16x8, uint4{pk[k][0], pk[k][1], pk[k][2], pk[k][3]});
}

// e^d for d <= 0 as 2^(d log2 e) on the hardware exp2 (0 for d = -inf)
__device__ __forceinline__ float exp_le0(float d) { return __builtin_amdgcn_exp2f(d * 1.44269504088896341f); }

// max and sum over the 32 lanes of a half-wave: the 16-lane DPP exchanges, then the other row's
// result through a swizzle (every lane ends with the same bits)
__device__ __forceinline__ float half32_max(float v) {
    v = row16_max_f(v);
    return maxf_bits(v, swz_xor16(__builtin_bit_cast(uint32_t, v)));
}
__device__ __forceinline__ float half32_sum(float v) {
    v = row16_sum_f(v);
    return v + __builtin_bit_cast(float, swz_xor16(__builtin_bit_cast(uint32_t, v)));
}

//
// With kin / vin set (one decode token, n_tok = 1) the kernel also stores that token's key and value
// rows: the workgroups whose chunk holds position p0 quantise them (bit for bit k_kv_store's Q8_0),
// head group 0 writes them to ring slot p0 % cap, and each writes them over the stale slot's copy
// in its LDS stage before computing it (the value scales of the stage's later keys, copies of that
// slot, are set to 0: those keys weigh 0).
template <int NB>
__global__ __launch_bounds__(ST_WAVES * 64) void k_attn_stream(
    const float *__restrict__ q, uint8_t *__restrict__ kc, uint8_t *__restrict__ vc, float *__restrict__ out,
    float *__restrict__ part, int n_tok, int n_head, int n_kv, int G, int p0, int cap, int window, int n_chunks,
    const float *__restrict__ kin, const float *__restrict__ vin) {
    using Sh = StreamShape<NB>;
    constexpr int HD = Sh::HD, SBW = Sh::SBW, VBW = Sh::VBW, PMASK = 2 * NB - 1;
    __shared__ __attribute__((aligned(16))) uint8_t ring[ST_RING * Sh::STAGE];
    __shared__ __attribute__((aligned(16))) float red[4 * 16 * ST_KEYS];  // [block quarter][head][key]
    __shared__ __attribute__((aligned(16))) float pl[16 * ST_PP];          // [head][key]: the stage's p
    __shared__ __attribute__((aligned(16))) float hcorr[16], hsum[16];
    const int lane = threadIdx.x & 63, lr = lane & 15, jg = lane >> 4, lk = lane & 31;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // workgroup -> (tile, head group) as in k_attn_split
    const int S = (n_head / n_kv) / G;
    const int xcd = blockIdx.x & 7, rest = blockIdx.x >> 3;
    const int sg = rest % S;
    const long T = (long)(rest / S) * 8 + xcd;
    if (T >= (long)n_tok * n_kv * n_chunks) return;
    const int c = (int)(T % n_chunks);
    const int tg = (int)(T / n_chunks);
    const int g = tg % n_kv, t = tg / n_kv;
    const int h0 = g * (n_head / n_kv) + sg * G;
    const int pos = p0 + t;
    const int lo = window > 0 ? max(0, pos + 1 - window) : 0;
    const int len = pos - lo + 1;
    const int per = (len + n_chunks - 1) / n_chunks;
    const int k0 = lo + c * per, k1 = min(pos + 1, k0 + per);
    const int nkeys = max(0, k1 - k0), nst = (nkeys + ST_KEYS - 1) / ST_KEYS;
    const size_t slot_bytes = (size_t)n_kv * Sh::ROW;
    const int slot0 = k0 % cap;
    const uint8_t *kg = kc + (size_t)g * Sh::ROW, *vg = vc + (size_t)g * Sh::ROW;

    // the copies of stage s into its ring slot. Every wave issues exactly NI copy instructions per
    // stage, stages past the tile included (those repeat one row, which stays in the caches), so that
    // the waits count stages; keys past the tile repeat its last key. Copy i of this lane: the key,
    // K or V, and the byte offset in the row are the same in every stage.
    int ckey[Sh::NI];
    const uint8_t *crow[Sh::NI];  // row base of the key's slot in stage 0, K or V
    uint32_t coff[Sh::NI];
#pragma unroll
    for (int i = 0; i < Sh::NQ; ++i) {
        const int P = (w * Sh::NQ + i) * 64 + lane;  // 16-byte slot of the stage: [K/V][key][slot]
        const int key = (P / (2 * NB)) % ST_KEYS, j = (P & PMASK) ^ (key & PMASK);  // the piece it holds
        ckey[i] = key;
        crow[i] = P / (64 * NB) ? vg : kg;
        coff[i] = Q8_BLOCK * (j >> 1) + 2 + 16 * (j & 1);
    }
#pragma unroll
    for (int i = 0; i < Sh::NS; ++i) {
        const int P = (w * Sh::NS + i) * 64 + lane;  // scale dword of the stage: [K/V][key][block]
        ckey[Sh::NQ + i] = (P / NB) % ST_KEYS;
        crow[Sh::NQ + i] = P / (32 * NB) ? vg : kg;
        coff[Sh::NQ + i] = Q8_BLOCK * (P % NB);  // the dword starting at the block's scale
    }
    const uint32_t ring0 = lds_addr(ring);
    auto issue = [&](int s) {
        const uint32_t base = ring0 + (s % ST_RING) * Sh::STAGE;
        const int kb = s * ST_KEYS;
        const uint8_t *src[Sh::NI];
        if (kb + ST_KEYS <= nkeys && slot0 + kb + ST_KEYS <= cap) {  // whole stage, no wrap
            const size_t adv = (size_t)(slot0 + kb) * slot_bytes;
#pragma unroll
            for (int i = 0; i < Sh::NI; ++i) src[i] = crow[i] + adv + ((size_t)ckey[i] * slot_bytes + coff[i]);
        } else {
            const bool real = s < nst;
            const int last = real ? min(ST_KEYS, nkeys - kb) - 1 : 0;
#pragma unroll
            for (int i = 0; i < Sh::NI; ++i) {
                int sl = slot0 + (real ? kb + min(ckey[i], last) : 0);
                sl = sl >= cap ? sl - cap : sl;
                src[i] = crow[i] + (size_t)sl * slot_bytes + coff[i];
            }
        }
#pragma unroll
        for (int i = 0; i < Sh::NQ; ++i) lds_copy16(src[i], base + (w * Sh::NQ + i) * 1024);
#pragma unroll
        for (int i = 0; i < Sh::NS; ++i)
            lds_copy4(src[Sh::NQ + i], base + Sh::QBYTES + (w * Sh::NS + i) * 256);
    };

    // the new token's key and value (fused store): half-wave (w, lane / 32) quantises blocks
    // 16 i + 2 w + lane / 32 of [K blocks, V blocks], element lane % 32
    constexpr int NPASS = NB / 8;
    const bool fuse = kin != nullptr && k0 <= pos && pos < k1;
    float fx[NPASS];
    if (fuse) {
#pragma unroll
        for (int i = 0; i < NPASS; ++i) {
            const int B = 16 * i + 2 * w + (lane >> 5);
            fx[i] = (B < NB ? kin : vin)[(size_t)g * HD + QK * (B % NB) + lk];
        }
    }

    // the queries and stage 0 first: 16 rows of HD floats (heads past G repeat head h0) into the last
    // ring slot, which the first stages leave free; stages 1 and 2 once those have landed, so that the
    // first stage of every workgroup is not queued behind the next ones
    {
        const uint32_t qbase = ring0 + (ST_RING - 1) * Sh::STAGE;
        const float *qrow = q + ((size_t)t * n_head + h0) * HD;
#pragma unroll
        for (int i = 0; i < Sh::NQ; ++i) {
            const int P = (w * Sh::NQ + i) * 64 + lane;  // 16-byte piece of the 16 x HD floats
            const int hh = P / (HD / 4), e = P % (HD / 4);
            lds_copy16(qrow + (size_t)(hh < G ? hh : 0) * HD + 4 * e, qbase + (w * Sh::NQ + i) * 1024);
        }
    }
    issue(0);
    __builtin_amdgcn_s_waitcnt(vmcnt_only(0));
    __syncthreads();
#pragma unroll
    for (int s = 1; s < ST_RING - 1; ++s) issue(s);
    // the fused token's row (its stores come after the copies of stages 1 and 2; the waits below
    // count loads, which complete in order, so a store still in flight only delays them)
    int fq[NPASS];
    uint16_t fd[NPASS];
    if (fuse) {
        uint8_t *slotp = nullptr;
        const int sp = p0 % cap;
#pragma unroll
        for (int i = 0; i < NPASS; ++i) {
            const int B = 16 * i + 2 * w + (lane >> 5);
            fq[i] = quant_q8_half(fx[i], &fd[i]);
            if (sg == 0) {  // the ring row, as k_kv_store writes it
                slotp = (B < NB ? kc : vc) + ((size_t)sp * n_kv + g) * Sh::ROW + Q8_BLOCK * (B % NB);
                slotp[2 + lk] = (uint8_t)(int8_t)fq[i];
                if (lk == 0) {
                    slotp[0] = (uint8_t)(fd[i] & 0xff);
                    slotp[1] = (uint8_t)(fd[i] >> 8);
                }
            }
        }
    }

    // the scores' share of this wave: key group kq, blocks SBW bq .. SBW bq + SBW - 1; q fragments
    // (A: head lr, elements 8 jg .. + 7 of each block) as three bf16 parts
    const int kq = w & 1, bq = w >> 1;
    bf16x8 qa[SBW][3];
    {
        const float *qs = (const float *)(ring + (ST_RING - 1) * Sh::STAGE);
#pragma unroll
        for (int i = 0; i < SBW; ++i) {
            const int b = SBW * bq + i;
            const bool qok = lr < G;
            const float4 *qr = (const float4 *)(qs + lr * HD + b * QK + 8 * jg);
            const float4 x0 = qr[0], x1 = qr[1];
            const float x[8] = {qok ? x0.x : 0.0f, qok ? x0.y : 0.0f, qok ? x0.z : 0.0f, qok ? x0.w : 0.0f,
                                qok ? x1.x : 0.0f, qok ? x1.y : 0.0f, qok ? x1.z : 0.0f, qok ? x1.w : 0.0f};
            split3_bf16(x, qa[i]);
        }
    }

    // the softmax of heads hw = 2 w + lane / 32, key lk: running max and sum
    const int hw = 2 * w + (lane >> 5);
    float m = -INFINITY, lsum = 0.0f;
    f32x4 acc[VBW][2];
#pragma unroll
    for (int i = 0; i < VBW; ++i) acc[i][0] = acc[i][1] = f32x4{0, 0, 0, 0};

    for (int s = 0; s < nst; ++s) {
        if (s > 0) {  // stage s + 1 stays in flight; stage 0 was waited for with the queries
            __builtin_amdgcn_s_waitcnt(vmcnt_only((ST_RING - 3) * Sh::NI));
            __syncthreads();  // the stage is in LDS for every wave; the slot of stage s - 2 is free
            issue(s + ST_RING - 2);
        }
        const uint8_t *sb = ring + (s % ST_RING) * Sh::STAGE;
        const uint32_t *scl = (const uint32_t *)(sb + Sh::QBYTES);
        const int nk = min(ST_KEYS, nkeys - s * ST_KEYS);
        if (fuse && s == (pos - k0) / ST_KEYS) {  // the stage holding the new token: its row into LDS
            uint8_t *st = ring + (s % ST_RING) * Sh::STAGE;
            uint32_t *stsc = (uint32_t *)(st + Sh::QBYTES);
            const int kp = (pos - k0) % ST_KEYS;
#pragma unroll
            for (int i = 0; i < NPASS; ++i) {
                const int B = 16 * i + 2 * w + (lane >> 5), which = B / NB, b = B % NB;
                const int slot = (2 * b + (lk >> 4)) ^ (kp & PMASK);
                st[((which * ST_KEYS + kp) * 2 * NB + slot) * 16 + (lk & 15)] = (uint8_t)(int8_t)fq[i];
                if (lk == 0) stsc[(which * ST_KEYS + kp) * NB + b] = fd[i];
            }
            // the later keys of the stage repeat the stale slot: a value scale of 0 keeps them finite
            const int dk = kp + 1 + (int)threadIdx.x / NB, db = (int)threadIdx.x % NB;
            if (dk < ST_KEYS) stsc[(ST_KEYS + dk) * NB + db] = 0u;
            __syncthreads();
        }

        // ---- scores: heads x keys 16 kq .. 16 kq + 15 over this wave's blocks
        if (kq == 0 || nk > 16) {
            const int kl = 16 * kq + lr;
            f32x4 s4 = {0, 0, 0, 0};
#pragma unroll
            for (int i = 0; i < SBW; ++i) {
                const int b = SBW * bq + i;
                const int slot = (2 * b + (jg >> 1)) ^ (kl & PMASK);
                const uint2 kw = *(const uint2 *)(sb + (kl * 2 * NB + slot) * 16 + 8 * (jg & 1));
                const bf16x8 bk = q8x8_bf16(kw.x, kw.y);
                f32x4 d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(qa[i][0], bk, f32x4{0, 0, 0, 0}, 0, 0, 0);
                d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(qa[i][1], bk, d, 0, 0, 0);
                d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(qa[i][2], bk, d, 0, 0, 0);
                const float dk = h2f((uint16_t)scl[kl * NB + b]);
#pragma unroll
                for (int r = 0; r < 4; ++r) s4[r] = fmaf(dk, d[r], s4[r]);
            }
            float *rw = red + bq * 16 * ST_KEYS;
#pragma unroll
            for (int r = 0; r < 4; ++r) rw[(4 * jg + r) * ST_KEYS + kl] = s4[r];
        }
        __syncthreads();

        // ---- online softmax of heads 2 w, 2 w + 1 over the stage's keys (one key per lane)
        {
            const int hh = hw < 16 ? hw : 0;
            float sv = ((red[hh * ST_KEYS + lk] + red[(16 + hh) * ST_KEYS + lk]) + red[(32 + hh) * ST_KEYS + lk]) +
                       red[(48 + hh) * ST_KEYS + lk];
            sv = lk < nk ? sv : -INFINITY;
            const float mn = fmaxf(m, half32_max(sv));
            const float corr = exp_le0(m - mn);  // 0 while m = -inf
            const float p = exp_le0(sv - mn);    // 0 for keys past the stage
            lsum = lsum * corr + half32_sum(p);
            m = mn;
            if (hw < 16) {
                pl[hw * ST_PP + lk] = hw < G ? p : 0.0f;
                if (lk == 0) hcorr[hw] = corr;
            }
        }
        __syncthreads();

        // ---- values: heads x the 32 dimensions of each of the wave's blocks
        {
            const float4 *pr = (const float4 *)(pl + lr * ST_PP + 8 * jg);
            const float4 pa = pr[0], pb = pr[1];
            const float p[8] = {pa.x, pa.y, pa.z, pa.w, pb.x, pb.y, pb.z, pb.w};
            const float4 cr = *(const float4 *)(hcorr + 4 * jg);  // rows 4 jg .. 4 jg + 3 of the MFMA output
#pragma unroll
            for (int i = 0; i < VBW; ++i)
#pragma unroll
                for (int tt = 0; tt < 2; ++tt) {
                    acc[i][tt][0] *= cr.x;
                    acc[i][tt][1] *= cr.y;
                    acc[i][tt][2] *= cr.z;
                    acc[i][tt][3] *= cr.w;
                }
#pragma unroll
            for (int i = 0; i < VBW; ++i) {
                const int b = w + ST_WAVES * i;
                float x[8];
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    x[e] = p[e] * h2f((uint16_t)scl[(ST_KEYS + 8 * jg + e) * NB + b]);
                bf16x8 a[3];
                split3_bf16(x, a);
#pragma unroll
                for (int tt = 0; tt < 2; ++tt) {
                    // source row of this lane: key 8 jg + lr / 2, dimensions 32 b + 16 tt + 8 (lr & 1) .. + 7
                    const int kl = 8 * jg + (lr >> 1);
                    const int slot = (2 * b + tt) ^ (kl & PMASK);
                    const uint8_t *src = sb + ((ST_KEYS + kl) * 2 * NB + slot) * 16 + 8 * (lr & 1);
                    const v2i_t vt = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_v2i_t *)src);
                    const bf16x8 bv = q8x8_bf16((uint32_t)vt.x, (uint32_t)vt.y);
                    acc[i][tt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[0], bv, acc[i][tt], 0, 0, 0);
                    acc[i][tt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[1], bv, acc[i][tt], 0, 0, 0);
                    acc[i][tt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[2], bv, acc[i][tt], 0, 0, 0);
                }
            }
        }
    }

    // the copies past the last stage land in LDS: none may be in flight when the workgroup ends
    __builtin_amdgcn_s_waitcnt(vmcnt_only(0));

    // ---- results: lane (lr, jg) holds heads 4 jg + r, dimension 32 b + 16 tt + lr of each block
    const size_t r0 = (size_t)t * n_head + h0;
    if (hw < 16 && lk == 0) hsum[hw] = lsum;
    __syncthreads();
    if (n_chunks == 1) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int h = 4 * jg + r;
            const float inv = 1.0f / hsum[h];
            if (h < G)
#pragma unroll
                for (int i = 0; i < VBW; ++i)
#pragma unroll
                    for (int tt = 0; tt < 2; ++tt)
                        out[(r0 + h) * HD + 32 * (w + ST_WAVES * i) + 16 * tt + lr] = acc[i][tt][r] * inv;
        }
    } else {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int h = 4 * jg + r;
            if (h < G) {
                float *pp = part + ((r0 + h) * n_chunks + c) * (size_t)(HD + 2);
#pragma unroll
                for (int i = 0; i < VBW; ++i)
#pragma unroll
                    for (int tt = 0; tt < 2; ++tt) pp[2 + 32 * (w + ST_WAVES * i) + 16 * tt + lr] = acc[i][tt][r];
            }
        }
        if (hw < G && lk == 0) {
            float *pp = part + ((r0 + hw) * n_chunks + c) * (size_t)(HD + 2);
            pp[0] = m;
            pp[1] = lsum;
        }
    }
}

// ---- Several tokens: 32 query rows of a kv head per workgroup ----
// Rows are (token, query head of the kv head) pairs, 32 per workgroup, so every key and value row is
// read once per 32 rows instead of once per token. A team of TW waves takes NBW * TW = NB blocks of
// the head dimension (NBW per wave); the 4 / TW teams of a workgroup take every (4 / TW)-th stage of
// 32 keys and merge once at the end. A wave copies its own blocks of the stage to LDS
// (global_load_lds) and reads nothing another wave copied, so the stages need no barrier; with
// TW = 2 the two waves of a team exchange their partial scores, one barrier per stage. The key copies
// of the next stage run under the softmax and the values, its value copies under the scores.
//
// Both products run on v_mfma_f32_32x32x16_f16, with the keys (the dimensions) as rows and the query
// rows as columns, so that a lane's accumulators all belong to its own query row (lane & 31): the
// softmax of a row is 16 values in each of two lanes, and its p are the B operand of the value
// product as they stand: the score product's row r holds key 16 (r / 4 % 2) + 4 (r / 8) + r % 4, so
// that register i of a lane is key 16 (lane / 32) + i, and the value product takes the keys in that
// order (its quants are read transposed, each lane group from its own keys).
//  - int8 quants are exact in f16;
//  - q times a power of two of its row (the row's largest lies in [2^14, 2^15)) is the sum of two
//    f16: 2^-23 of the element, or 2^-39 of the row's largest for smaller ones;
//  - p 2^10 likewise, once per stage (p down to 2^-24 has 11 bits or more); a block's p d_v is then
//    formed in f16 pairs, hi = ph d_v rounded and lo = pl d_v + (ph d_v - hi), whose bracket is exact (a
//    product of two 11-bit numbers). d_v enters as d_v 2^-E, E the exponent of the largest scale of the
//    stages so far: exact down to 2^-14 of 2^E, and p d_v to 2^-33 of 2^E.
// The last is too little for a row whose own scales lie far below 2^E (another block's, a key's that weighs
// nothing in it or that it does not see), as 2^-39 of a row's q is for a block of it that meets large key scales.
// So a wave keeps the smallest scale too, and where one of a workgroup's waves met a 0 or a scale under
// 2^(E - PF_NEAR), or a block of q under 2^-PF_Q of its row, the workgroup walks its stages again: such a
// block of q has a power of two of its own (2^-23 of the block's largest throughout), and p d_v is formed in f32
// and scaled by its own power of two per row, block and stage: f16 pairs of 2^-23 of a product, or 2^-39 of
// the row's largest in the stage. (Both walks, 512 tokens in a window of 1024 keys: 101 us, 53 for one in the
// same run; 500 tokens x 16 heads of 512 on 4,100 keys 583, 247 for one. The pairs of the second walk in every
// stage of a single one would cost that much always, and a branch per stage 2 to 5% of the first.)
// Two waves share a SIMD (at most 256 registers: 4 blocks per wave; 8 blocks per wave and one wave per
// SIMD took 356 us against 274 on hd 512, the waits of one wave having nothing beside them). What bounds
// it: VALU, about 620 instructions per wave and stage of 4 blocks against 32 MFMAs. Per workgroup and
// round of stages 3.9 us (500 tokens x 16 heads of 512 on 3,601 to 4,100 keys, 247 us, 257 TFLOP/s of
// the two products; per-token kernel 1244 us); without the copies 3.4 us.
constexpr int PF_ROWS = 32, PF_KEYS = 32;
// With every scale in [2^(E - 11), 2^(E + 1)) the key of a row's largest weight (p >= 1/2) has a p d_v of at least
// 2^(E - 12), and what the other keys' may miss, 2^-33 2^E, is 2^-21 of that.
constexpr int PF_NEAR = 11, PF_Q = 16;
// the binary16 bits of 2^(E - PF_NEAR), E >= -15 (1, the smallest scale, if that is below it)
__device__ __forceinline__ uint32_t pf_near_bits(int E) {
    const int e = E - PF_NEAR;
    return e >= -14 ? (uint32_t)(e + 15) << 10 : e >= -24 ? 1u << (e + 24) : 1u;
}

typedef float f32x16 __attribute__((ext_vector_type(16)));

template <int NBW, int TW, int WV>
struct PrefillShape {
    static constexpr int NB = NBW * TW, HD = 32 * NB, ROW = NB * Q8_BLOCK, NT = WV / TW;
    static constexpr int NQ = NBW, NS = NBW / 2, NI = NQ + NS;  // 16- and 4-byte copies of a wave's K or V stage
    static constexpr int QBYTES = NBW * 1024, SBYTES = NBW * 128;
    static constexpr int WAVE = 2 * QBYTES + 2 * SBYTES + 2 * NBW * 64;  // quants, scale dwords, packed scales
    static constexpr int XCHG = TW > 1 ? 2 * WV * 4096 : 0;    // partial scores, two buffers
    static constexpr int MERGE = WV * NBW * 16 * 256;          // the waves' value sums
    static constexpr int LOOP = WV * WAVE + XCHG;
    static constexpr int LDS = LOOP > MERGE ? LOOP : MERGE;
    static_assert(LDS + 4096 <= 163840, "LDS");
};

// 16 (4) bytes per lane at base + off to LDS (see lds_copy16), base the same in every lane
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void lds_copy16_at(const void *base, uint32_t off, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(off), "s"(base), "s"(lds) : "memory", "m0");
}
__device__ __forceinline__ void lds_copy4_at(const void *base, uint32_t off, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dword %0, %1" : : "v"(off), "s"(base), "s"(lds) : "memory", "m0");
}
#pragma clang diagnostic pop
// every LDS operation of this wave has completed
__device__ __forceinline__ void lds_done() { asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory"); }
template <int N>
__device__ __forceinline__ void loads_left() {  // at most N vector memory operations are in flight
    asm volatile("s_waitcnt vmcnt(%0)" : : "n"(N) : "memory");
}

// eight int8 quants as f16: 0x6400 | (q + 128) is 1152 + q
__device__ __forceinline__ f16x8 q8x8_f16(uint32_t a, uint32_t b) {
    const f16x2 off = {(_Float16)1152.0f, (_Float16)1152.0f};
    a ^= 0x80808080u;
    b ^= 0x80808080u;
    uint32_t u[4];
    u[0] = as_u32(as_f16x2(__builtin_amdgcn_perm(0x64646464u, a, 0x04010400u)) - off);
    u[1] = as_u32(as_f16x2(__builtin_amdgcn_perm(0x64646464u, a, 0x04030402u)) - off);
    u[2] = as_u32(as_f16x2(__builtin_amdgcn_perm(0x64646464u, b, 0x04010400u)) - off);
    u[3] = as_u32(as_f16x2(__builtin_amdgcn_perm(0x64646464u, b, 0x04030402u)) - off);
    return as_f16x8(u);
}

struct __attribute__((packed, aligned(4))) F4u {  // four floats on any dword
    float v[4];
};

template <int NBW, int TW, int WV>
__global__ __launch_bounds__(WV * 64) void k_attn_prefill(
    const float *__restrict__ q, const uint8_t *__restrict__ kc, const uint8_t *__restrict__ vc,
    float *__restrict__ out, float *__restrict__ part, int n_tok, int n_head, int n_kv, int p0, int cap, int window,
    int n_chunks, int tiles) {
    using Sh = PrefillShape<NBW, TW, WV>;
    constexpr int HD = Sh::HD, NT = Sh::NT, PM = 2 * NBW - 1;
    constexpr float LOG2E = 1.44269504088896341f;
    constexpr int PK = 10;  // p <= 2^4 and d_v 2^-E < 2: p 2^PK d_v 2^-E < 2^15
    __shared__ __attribute__((aligned(1024))) uint8_t sh[Sh::LDS];
    __shared__ float wm[NT][PF_ROWS], wt[NT][PF_ROWS], wl[NT][PF_ROWS], wmax[WV][PF_ROWS], wus[WV];
    __shared__ int wapart[WV], qdiff[WV][NBW][PF_ROWS];
    const int lane = threadIdx.x & 63, lr = lane & 31, hf = lane >> 5;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int team = w / TW, pw = w % TW;  // blocks NBW pw .. NBW pw + NBW - 1 of the team's stages
    // workgroup -> (kv head, chunk, tile of rows): the kv head varies fastest, so that with 2, 4 or 8
    // of them each XCD's L2 serves one; the last tokens (the most keys) start first
    const int HG = n_head / n_kv, rows = n_tok * HG;
    const int g = blockIdx.x % n_kv, rest = blockIdx.x / n_kv;
    const int c = rest % n_chunks, tile = tiles - 1 - rest / n_chunks;
    const int row = tile * PF_ROWS + lr, rc = min(row, rows - 1);  // rows past the last repeat it, unstored
    const int t = rc / HG, h = g * HG + rc % HG;
    // the row's keys [k0, k1): both bounds grow with the token
    const int pos = p0 + t;
    const int lo = window > 0 ? max(0, pos + 1 - window) : 0;
    const int per = (pos - lo + 1 + n_chunks - 1) / n_chunks;
    const int k0 = lo + c * per, k1 = k0 + min(per, pos + 1 - k0);
    const int u0 = __builtin_amdgcn_readlane(k0, 0), u1 = __builtin_amdgcn_readlane(k1, 31);  // any row's
    const int f0 = __builtin_amdgcn_readlane(k0, 31), f1 = __builtin_amdgcn_readlane(k1, 0);  // every row's
    const int nst = u1 > u0 ? (u1 - u0 + PF_KEYS - 1) / PF_KEYS : 0, nit = (nst + NT - 1) / NT;

    uint8_t *const kq = sh + w * Sh::WAVE, *const vq = kq + Sh::QBYTES;
    uint8_t *const ks = vq + Sh::QBYTES, *const vs = ks + Sh::SBYTES, *const ksp = vs + Sh::SBYTES,
            *const vsp = ksp + NBW * 64;
    const size_t slot_bytes = (size_t)n_kv * Sh::ROW;
    const uint8_t *kg = kc + (size_t)g * Sh::ROW + pw * NBW * Q8_BLOCK;
    const uint8_t *vg = vc + (size_t)g * Sh::ROW + pw * NBW * Q8_BLOCK;
    // a stage's copies: quants as [key][16-byte piece p ^ swz(key)], the scales as the dwords that start
    // at them, [block][key]. swz puts what 16 lanes read at once on distinct banks: one piece of keys
    // 0 .. 7 and 16 .. 23 (8 .. 15 and 24 .. 31), and two pieces of eight keys
    auto swz = [](int key) {
        return NBW == 2 ? (key >> 1 & 2) | (key >> 4 & 1) : (key ^ (key >> 4 & 1)) & PM;
    };
    auto copy_key = [&](int i) { return (i * 64 + lane) / (2 * NBW); };
    auto copy_off = [&](int i) {
        const int piece = (lane & PM) ^ swz(copy_key(i));
        return Q8_BLOCK * (piece >> 1) + 2 + 16 * (piece & 1);
    };
    uint32_t qoff[Sh::NQ], soff[Sh::NS];
#pragma unroll
    for (int i = 0; i < Sh::NQ; ++i) qoff[i] = (uint32_t)copy_key(i) * (uint32_t)slot_bytes + copy_off(i);
#pragma unroll
    for (int i = 0; i < Sh::NS; ++i) soff[i] = (uint32_t)lr * (uint32_t)slot_bytes + Q8_BLOCK * (2 * i + hf);
    auto issue = [&](const uint8_t *base, uint32_t dq, uint32_t ds, int key0) {
        const int s0 = key0 % cap;
        const int last = u1 - 1 - key0;  // (positions reach 2^31 - 1: here and below key0 + 32 may not fit an int)
        if (last >= PF_KEYS - 1 && s0 + PF_KEYS <= cap) {  // a whole stage without a wrap
            const uint8_t *b = base + (size_t)s0 * slot_bytes;
#pragma unroll
            for (int i = 0; i < Sh::NQ; ++i) lds_copy16_at(b, qoff[i], dq + i * 1024);
#pragma unroll
            for (int i = 0; i < Sh::NS; ++i) lds_copy4_at(b, soff[i], ds + i * 256);
        } else {  // keys past the last repeat it
#pragma unroll 1
            for (int i = 0; i < Sh::NQ; ++i) {
                const int sl = (int)((uint32_t)(key0 + min(copy_key(i), last)) % (uint32_t)cap);
                lds_copy16(base + (size_t)sl * slot_bytes + copy_off(i), dq + i * 1024);
            }
            const int sl = (int)((uint32_t)(key0 + min(lr, last)) % (uint32_t)cap);
#pragma unroll 1
            for (int i = 0; i < Sh::NS; ++i)
                lds_copy4(base + (size_t)sl * slot_bytes + Q8_BLOCK * (2 * i + hf), ds + i * 256);
        }
    };
    const uint32_t akq = lds_addr(kq), avq = lds_addr(vq), aks = lds_addr(ks), avs = lds_addr(vs);
    auto first_copies = [&]() __attribute__((always_inline)) {
        if (team >= nst) return;
        issue(kg, akq, aks, u0 + team * PF_KEYS);
        issue(vg, avq, avs, u0 + team * PF_KEYS);
    };
    first_copies();

    // ---- q: the row's elements 32 b + 16 hf + 8 m .. + 7 of block b are MFMA m's K slots 8 hf ..
    f16x8 qh[NBW][2], ql[NBW][2];
    int qe;       // q is scaled by 2^qe,
    bool qapart;  // block b of some rows by 2^(qe - qdiff[w][b][row])
    {
        const float *qr = q + ((size_t)t * n_head + h) * HD + 32 * NBW * pw + 16 * hf;
        float mx = 0.0f, mb[NBW];
        F4u f[4 * NBW];
#pragma unroll
        for (int i = 0; i < 4 * NBW; ++i) f[i] = *(const F4u *)(qr + 32 * (i / 4) + 4 * (i % 4));
#pragma unroll
        for (int b = 0; b < NBW; ++b) {
            mb[b] = 0.0f;
#pragma unroll
            for (int i = 4 * b; i < 4 * b + 4; ++i)
#pragma unroll
                for (int e = 0; e < 4; ++e) mb[b] = fmaxf(mb[b], fabsf(f[i].v[e]));
            mb[b] = fmaxf(mb[b], __shfl_xor(mb[b], 32));
            mx = fmaxf(mx, mb[b]);
        }
        if constexpr (TW > 1) {  // the row's largest, over the team's waves
            if (hf == 0) wmax[w][lr] = mx;
            __syncthreads();
#pragma unroll
            for (int i = 0; i < TW; ++i) mx = fmaxf(mx, wmax[team * TW + i][lr]);
        }
        // mx 2^qe in [2^14, 2^15); under 2^-86, where every score is 0 to f32, 2^qe stays at 2^100
        auto up = [](float top) { return min(100, 14 + 127 - (int)((__float_as_uint(top) >> 23) & 0xFF)); };
        qe = up(mx);
        bool low = false;
#pragma unroll
        for (int b = 0; b < NBW; ++b) low |= mb[b] > 0.0f && mb[b] < ldexpf(mx, -PF_Q);
        qapart = __builtin_amdgcn_ballot_w64(low) != 0;
#pragma unroll
        for (int b = 0; b < NBW; ++b) {
            int qb = qe;
            if (qapart) {
                if (mb[b] > 0.0f && mb[b] < ldexpf(mx, -PF_Q)) qb = up(mb[b]);
                qdiff[w][b][lr] = qe - qb;
            }
#pragma unroll
            for (int m = 0; m < 2; ++m) {
                uint32_t hi[4], lw[4];
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    const float *v = f[4 * b + 2 * m + u].v;
#pragma unroll
                    for (int e = 0; e < 2; ++e) {
                        f16x2 a, r;
                        split2_f16(ldexpf(v[2 * e], qb), ldexpf(v[2 * e + 1], qb), a, r);
                        hi[2 * u + e] = as_u32(a);
                        lw[2 * u + e] = as_u32(r);
                    }
                }
                qh[b][m] = as_f16x8(hi);
                ql[b][m] = as_f16x8(lw);
            }
            if (b % 2) __builtin_amdgcn_sched_barrier(0);
        }
    }
    const float L = ldexpf(LOG2E, -qe);  // scores are in units of 2^-qe; times L: log2 of their exponential

    // the row's largest score, the reference m that p is relative to (p = 2^(score L - m)), and the sum
    // of p 2^PK over this lane's keys (its other half: lane ^ 32)
    float mt, m, l;
    int E;          // exponent of the largest value scale so far
    uint32_t dlow;  // the bits of the smallest of this lane's copies of them
    f32x16 acc[NBW];
    // LDS offsets of this lane's first key quants and value quants (block 0; block b: ^ 32 b, as a
    // row of 32 NBW bytes is aligned to its size)
    uint32_t kra, vra;
    {
        const int key = 16 * ((lr >> 2) & 1) + 4 * (lr >> 3) + (lr & 3);
        kra = w * Sh::WAVE + (key * 2 * NBW + (hf ^ swz(key))) * 16;
    }
    {
        // the transposed read: a group of 16 lanes takes 8 keys x 16 dimensions
        const int key = 16 * hf + ((lane & 15) >> 1);
        vra = w * Sh::WAVE + Sh::QBYTES + (key * 2 * NBW + (((lane >> 4) & 1) ^ swz(key))) * 16 + 8 * (lane & 1);
    }

    // every stage of the team; APART: p d_v in f32 (above)
    auto walk = [&](auto apart) __attribute__((always_inline)) {
        constexpr bool APART = decltype(apart)::value;
        mt = m = -INFINITY;
        l = 0.0f;
        E = -15;
        dlow = 0x7FFFu;
#pragma unroll
        for (int b = 0; b < NBW; ++b)
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[b][i] = 0.0f;
        for (int it = 0; it < nit; ++it) {
            const int s = it * NT + team;
            const bool live = s < nst, next = s + NT < nst;
            const int key0 = u0 + s * PF_KEYS;
            if (!live) {  // a team past its last stage keeps the barriers
                if constexpr (TW > 1) __builtin_amdgcn_s_barrier();
                continue;
            }
            f32x16 sc;
            asm volatile("" : "+v"(kra), "+v"(vra));  // the blocks' offsets are formed where they are used
            // ---- scores: sc[i] = key 16 hf + i of the stage, query row lr
            loads_left<Sh::NI>();  // the keys are in LDS (the values may be in flight)
            // a block's key quants and scales are read one block ahead of their use, and its scale
            // products run under the next block's MFMAs
            uint4 kw = *(const uint4 *)(sh + kra);
#pragma unroll
            for (int i = 0; i < Sh::NS; ++i)
                *(uint16_t *)(ksp + ((2 * i + hf) * 32 + lr) * 2) =
                    (uint16_t)*(const uint32_t *)(ks + (64 * i + lane) * 4);
            wave_lds_sync();
            f32x16 dp;
#pragma unroll
            for (int i = 0; i < 16; ++i) sc[i] = 0.0f;
            uint4 dk[2];
            auto scale = [&](f32x16 &d, const uint4 (&k)[2], int b) {
                if (APART && qapart) {
                    const int by = qdiff[w][b][lr];
#pragma unroll
                    for (int i = 0; i < 16; ++i) d[i] = ldexpf(d[i], by);
                }
                const uint32_t dw[8] = {k[0].x, k[0].y, k[0].z, k[0].w, k[1].x, k[1].y, k[1].z, k[1].w};
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    sc[2 * e] = fmaf((float)as_f16x2(dw[e]).x, d[2 * e], sc[2 * e]);
                    sc[2 * e + 1] = fmaf((float)as_f16x2(dw[e]).y, d[2 * e + 1], sc[2 * e + 1]);
                }
                asm volatile("" : "+v"(sc));  // here, and not where the sums are used
            };
#pragma unroll
            for (int b = 0; b < NBW; ++b) {
                const uint4 kn = b + 1 < NBW ? *(const uint4 *)(sh + (kra ^ (32 * (b + 1)))) : kw;
                const uint4 *dq = (const uint4 *)(ksp + b * 64 + 32 * hf);
                const uint4 dn[2] = {dq[0], dq[1]};
                const f16x8 a0 = q8x8_f16(kw.x, kw.y), a1 = q8x8_f16(kw.z, kw.w);
                f32x16 d;
#pragma unroll
                for (int i = 0; i < 16; ++i) d[i] = 0.0f;
                d = __builtin_amdgcn_mfma_f32_32x32x16_f16(a0, ql[b][0], d, 0, 0, 0);
                d = __builtin_amdgcn_mfma_f32_32x32x16_f16(a1, ql[b][1], d, 0, 0, 0);
                d = __builtin_amdgcn_mfma_f32_32x32x16_f16(a0, qh[b][0], d, 0, 0, 0);
                d = __builtin_amdgcn_mfma_f32_32x32x16_f16(a1, qh[b][1], d, 0, 0, 0);
                if (b > 0) scale(dp, dk, b - 1);
                dp = d;
                kw = kn;
                dk[0] = dn[0];
                dk[1] = dn[1];
                __builtin_amdgcn_sched_barrier(0);
            }
            scale(dp, dk, NBW - 1);
            lds_done();
            if (next) issue(kg, akq, aks, key0 + NT * PF_KEYS);
            if constexpr (TW > 1) {  // both waves of a team add the same two partial scores
                float4 *x = (float4 *)(sh + WV * Sh::WAVE) + (it & 1) * WV * 256 + lane;
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    x[w * 256 + 64 * i] = make_float4(sc[4 * i], sc[4 * i + 1], sc[4 * i + 2], sc[4 * i + 3]);
                lds_done();
                __builtin_amdgcn_s_barrier();
                asm volatile("" : : : "memory");
#pragma unroll
                for (int i = 0; i < 4; ++i) {  // (0 + 1) + (2 + 3)
                    const float4 o = x[(w ^ 1) * 256 + 64 * i];
                    sc[4 * i] += o.x;
                    sc[4 * i + 1] += o.y;
                    sc[4 * i + 2] += o.z;
                    sc[4 * i + 3] += o.w;
                    if constexpr (TW == 4) {
                        const float4 u = x[(w ^ 2) * 256 + 64 * i], v = x[(w ^ 3) * 256 + 64 * i];
                        sc[4 * i] += u.x + v.x;
                        sc[4 * i + 1] += u.y + v.y;
                        sc[4 * i + 2] += u.z + v.z;
                        sc[4 * i + 3] += u.w + v.w;
                    }
                }
            }
            // ---- online softmax of the row
            const bool whole = key0 >= f0 && f1 - key0 >= PF_KEYS;  // no key masked for any row
            uint32_t seen = 0xFFFFu;
            if (!whole) {
                seen = 0;
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    const uint32_t key = (uint32_t)key0 + 16 * hf + i;
                    const bool in = key >= (uint32_t)k0 && key < (uint32_t)k1;
                    seen |= in ? 1u << i : 0u;
                    sc[i] = in ? sc[i] : -INFINITY;
                }
            }
            float mx = sc[0];
#pragma unroll
            for (int i = 1; i < 16; ++i) mx = fmaxf(mx, sc[i]);
            mx = fmaxf(mx, __shfl_xor(mx, 32));
            mt = fmaxf(mt, mx);

            // ---- the stage's value scales: their largest, then d_v 2^-E packed as [block][key]
            if (next) loads_left<Sh::NI>();
            else loads_left<0>();
            uint32_t dbits[Sh::NS], dmax = 0, nonfin = 0;
#pragma unroll
            for (int i = 0; i < Sh::NS; ++i) {
                dbits[i] = *(const uint32_t *)(vs + (64 * i + lane) * 4) & 0xFFFFu;
                const uint32_t mag = dbits[i] & 0x7FFFu;
                nonfin |= mag >= 0x7C00u ? 1u : 0u;
                dmax = max(dmax, mag >= 0x7C00u ? 0u : mag);
                if constexpr (!APART) dlow = min(dlow, mag);
            }
            const int dtop = (int)half32_max((float)dmax);
            const int En =
                max(E, (max(__builtin_amdgcn_readlane(dtop, 0), __builtin_amdgcn_readlane(dtop, 32)) >> 10) - 15);
            // the reference m, a whole number (so that every rescale is exact), moves only when a score
            // passes it by more than 4 (in log2): p <= 16
            float corr = ldexpf(1.0f, E - En);
            E = En;
            const float ml = mt * L;
            if (__builtin_amdgcn_ballot_w64(ml - m > 4.0f || m == -INFINITY)) {
                const float up = ceilf(ml);
                const float f = up == -INFINITY ? 1.0f : __builtin_amdgcn_exp2f(m - up);  // 0 while m = -inf
                m = up;
                corr *= f;
                l *= f;
            }
#pragma unroll
            for (int i = 0; i < Sh::NS; ++i) {  // infinite and NaN scales are added below
                const bool fin = (dbits[i] & 0x7C00u) != 0x7C00u;
                *(_Float16 *)(vsp + ((2 * i + hf) * 32 + lr) * 2) =
                    (_Float16)(fin ? ldexpf(h2f((uint16_t)dbits[i]), APART ? 0 : -E) : 0.0f);
            }
            if (__builtin_amdgcn_ballot_w64(corr != 1.0f)) {
#pragma unroll
                for (int b = 0; b < NBW; ++b)
#pragma unroll
                    for (int i = 0; i < 16; ++i) acc[b][i] *= corr;
            }
            // p 2^PK, from a reference PK lower
            const float mr = (float)PK - (m == -INFINITY ? 0.0f : m);
            float ps = 0.0f;
            f16x2 ph[8], pl[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                sc[2 * i] = __builtin_amdgcn_exp2f(fmaf(sc[2 * i], L, mr));
                sc[2 * i + 1] = __builtin_amdgcn_exp2f(fmaf(sc[2 * i + 1], L, mr));
                ps += sc[2 * i] + sc[2 * i + 1];
                split2_f16(sc[2 * i], sc[2 * i + 1], ph[i], pl[i]);
            }
            l += ps;
            wave_lds_sync();
            if (__builtin_amdgcn_ballot_w64(nonfin)) {
                uint32_t sk = 0, pk = 0;  // this row's keys by stage position: seen, and of weight above 0
#pragma unroll
                for (int i = 0; i < 16; ++i) pk |= sc[i] > 0.0f ? 1u << i : 0u;
                sk = seen << (16 * hf);
                pk <<= 16 * hf;
                sk |= (uint32_t)__shfl_xor((int)sk, 32);
                pk |= (uint32_t)__shfl_xor((int)pk, 32);
#pragma unroll
                for (int b = 0; b < NBW; ++b)
#pragma unroll 1
                    for (int key = 0; key < PF_KEYS; ++key) {
                        const uint32_t db = *(const uint32_t *)(vs + (32 * b + key) * 4) & 0xFFFFu;
                        if ((db & 0x7C00u) != 0x7C00u) continue;
                        const float d = sk >> key & 1 ? (pk >> key & 1 ? h2f((uint16_t)db) : NAN) : 0.0f;
#pragma unroll
                        for (int i4 = 0; i4 < 4; ++i4) {  // quants of dimensions 8 i4 + 4 hf .. + 3
                            const int piece = (2 * b + (i4 >> 1)) ^ swz(key);
                            const uint32_t u =
                                *(const uint32_t *)(vq + (key * 2 * NBW + piece) * 16 + 8 * (i4 & 1) + 4 * hf);
#pragma unroll
                            for (int e = 0; e < 4; ++e) {
                                const float add = d * q8_at(u, e);
                                acc[b][4 * i4 + e] += sk >> key & 1 ? add : 0.0f;
                            }
                        }
                    }
            }

            // ---- values: acc[b][i] = dimension 32 b + 8 (i / 4) + 4 hf + i % 4, query row lr
            v2i_t vt[2];
            uint4 dv[2];
            auto read_quants = [&](int b, v2i_t (&vv)[2]) {
                const uint8_t *src = sh + (vra ^ (32 * b));
                vv[0] = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_v2i_t *)src);
                vv[1] = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_v2i_t *)(src + 256 * NBW));  // 8 keys on
            };
            if constexpr (APART) {
#pragma unroll
                for (int b = 0; b < NBW; ++b) {
                    // the products of keys 4 n .. 4 n + 3 of the lane's 16, formed twice instead of held
                    float wv[4];
                    auto products = [&](int n) {
                        asm volatile("" : : : "memory");
                        const uint2 r = *(const uint2 *)(vsp + b * 64 + 32 * hf + 8 * n);
                        const f16x2 d0 = as_f16x2(r.x), d1 = as_f16x2(r.y);
                        wv[0] = sc[4 * n] * (float)d0.x;
                        wv[1] = sc[4 * n + 1] * (float)d0.y;
                        wv[2] = sc[4 * n + 2] * (float)d1.x;
                        wv[3] = sc[4 * n + 3] * (float)d1.y;
                    };
                    float top = 0.0f, sum = 0.0f;
#pragma unroll
                    for (int n = 0; n < 4; ++n) {
                        products(n);
#pragma unroll
                        for (int e = 0; e < 4; ++e) top = fmaxf(top, fabsf(wv[e]));
                    }
#pragma unroll
                    for (int i = 0; i < 16; ++i) sum = fmaxf(sum, fabsf(acc[b][i]));
                    // times 2^up the products lie under 2^15, the sums so far under 2^100, in both of the row's lanes
                    int up = min(141 - (int)((__float_as_uint(top) >> 23) & 0xFF),
                                 226 - E - (int)((__float_as_uint(sum) >> 23) & 0xFF));
                    up = min(up, __shfl_xor(up, 32));
#pragma unroll
                    for (int i = 0; i < 16; ++i) acc[b][i] = ldexpf(acc[b][i], up + E);
                    read_quants(b, vt);
#pragma unroll
                    for (int mm = 0; mm < 2; ++mm) {
                        uint32_t bh[4], bl[4];
#pragma unroll
                        for (int x = 0; x < 4; ++x) {
                            if (x % 2 == 0) products(2 * mm + x / 2);
                            f16x2 hi, lw;
                            split2_f16(ldexpf(wv[2 * (x % 2)], up), ldexpf(wv[2 * (x % 2) + 1], up), hi, lw);
                            bh[x] = as_u32(hi);
                            bl[x] = as_u32(lw);
                        }
                        const f16x8 a = q8x8_f16((uint32_t)vt[mm].x, (uint32_t)vt[mm].y);
                        acc[b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, as_f16x8(bl), acc[b], 0, 0, 0);
                        acc[b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, as_f16x8(bh), acc[b], 0, 0, 0);
                        __builtin_amdgcn_sched_barrier(0);
                    }
#pragma unroll
                    for (int i = 0; i < 16; ++i) acc[b][i] = ldexpf(acc[b][i], -up - E);
                    __builtin_amdgcn_sched_barrier(0);
                }
            } else {
                auto read_values = [&](int b, v2i_t (&vv)[2], uint4 (&dd)[2]) {
                    read_quants(b, vv);
                    const uint4 *dq = (const uint4 *)(vsp + b * 64 + 32 * hf);
                    dd[0] = dq[0];
                    dd[1] = dq[1];
                };
                read_values(0, vt, dv);
#pragma unroll
                for (int b = 0; b < NBW; ++b) {
                    v2i_t vn[2] = {vt[0], vt[1]};
                    uint4 dn[2] = {dv[0], dv[1]};
                    if (b + 1 < NBW) read_values(b + 1, vn, dn);
                    f16x8 a[2];
                    uint32_t bh[2][4], bl[2][4];
#pragma unroll
                    for (int mm = 0; mm < 2; ++mm) {
                        a[mm] = q8x8_f16((uint32_t)vt[mm].x, (uint32_t)vt[mm].y);
                        const uint32_t dw[4] = {dv[mm].x, dv[mm].y, dv[mm].z, dv[mm].w};
#pragma unroll
                        for (int x = 0; x < 4; ++x) {
                            const f16x2 d2 = as_f16x2(dw[x]), hi = ph[4 * mm + x] * d2;
                            bh[mm][x] = as_u32(hi);
                            bl[mm][x] = as_u32(__builtin_elementwise_fma(
                                pl[4 * mm + x], d2, __builtin_elementwise_fma(ph[4 * mm + x], d2, -hi)));
                        }
                    }
                    acc[b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[0], as_f16x8(bl[0]), acc[b], 0, 0, 0);
                    acc[b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[1], as_f16x8(bl[1]), acc[b], 0, 0, 0);
                    acc[b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[0], as_f16x8(bh[0]), acc[b], 0, 0, 0);
                    acc[b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[1], as_f16x8(bh[1]), acc[b], 0, 0, 0);
                    vt[0] = vn[0];
                    vt[1] = vn[1];
                    dv[0] = dn[0];
                    dv[1] = dn[1];
                    if (b % 2) __builtin_amdgcn_sched_barrier(0);
                }
            }
            lds_done();
            if (next) issue(vg, avq, avs, key0 + NT * PF_KEYS);
        }
    };
    walk(std::false_type{});
    const bool apart = qapart || __builtin_amdgcn_ballot_w64(dlow < pf_near_bits(E)) != 0;
    if (lane == 0) wapart[w] = apart;
    __syncthreads();  // every wave is done with its stages
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(wapart[lane % WV] != 0) != 0, 0)) {
        first_copies();
        walk(std::true_type{});
        __syncthreads();
    }

    // ---- the teams' results meet in LDS: M = max of their maxima, the sums weighted by e^(m - M);
    // wave (team, pw) finishes a share of its blocks' registers
    l += __shfl_xor(l, 32);
    float *mrg = (float *)sh;  // [wave][block, register][lane]
#pragma unroll
    for (int b = 0; b < NBW; ++b)
#pragma unroll
        for (int i = 0; i < 16; ++i) mrg[((w * NBW + b) * 16 + i) * 64 + lane] = acc[b][i];
    if (lane == 0) wus[w] = ldexpf(1.0f, E - PK);
    if (pw == 0 && hf == 0) {
        wm[team][lr] = m;
        wt[team][lr] = mt * L;
        wl[team][lr] = ldexpf(l, -PK);
    }
    __syncthreads();
    float M = wm[0][lr], T = wt[0][lr], f[NT], den = 0.0f;
#pragma unroll
    for (int u = 1; u < NT; ++u) {
        M = fmaxf(M, wm[u][lr]);
        T = fmaxf(T, wt[u][lr]);
    }
    // a partial is relative to the natural logarithm of its largest weight, tn as rounded
    const float tn = T * 0.693147180559945309f;
    float to = 1.0f;
    if (n_chunks > 1 && fabsf(T) < INFINITY)
        to = __builtin_amdgcn_exp2f((M - T) + fmaf(tn, -1.92596299e-8f, fmaf(tn, -LOG2E, T)));
#pragma unroll
    for (int u = 0; u < NT; ++u) {
        f[u] = wm[u][lr] == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(wm[u][lr] - M) * to;
        den = fmaf(f[u], wl[u][lr], den);
        f[u] *= wus[u * TW + pw];
    }
    const float inv = n_chunks == 1 ? 1.0f / den : 1.0f;
    const size_t r0 = (size_t)t * n_head + h;
    float *dst = n_chunks == 1 ? out + r0 * HD : part + (r0 * n_chunks + c) * (size_t)(HD + 2) + 2;
    if (row >= rows) return;
    if (n_chunks > 1 && w == 0 && hf == 0) {
        dst[-2] = tn;
        dst[-1] = den;
    }
    constexpr int R4 = NBW * 4 / NT;  // groups of 4 registers per wave
#pragma unroll
    for (int r = 0; r < R4; ++r) {
        const int r4 = team * R4 + r;
        F4u o;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            float num = 0.0f;
#pragma unroll
            for (int u = 0; u < NT; ++u) num = fmaf(f[u], mrg[((u * TW + pw) * NBW * 16 + 4 * r4 + e) * 64 + lane], num);
            o.v[e] = num * inv;
        }
        *(F4u *)(dst + 32 * (NBW * pw + r4 / 4) + 8 * (r4 % 4) + 4 * hf) = o;
    }
}

// out[i][d] = sum_c e^(m_c - M) acc_c[d] / sum_c e^(m_c - M) l_c with M = max_c m_c; an empty chunk
// (m = -inf, l = 0) adds nothing (the reference's merge, runtime/hip/rvhip.hip:376-394).
// Workgroup (row, 64 dimensions), lane = dimension: wave w folds chunks w, w + 4, ... in one pass
// with a running maximum (rescaling what it holds when the maximum grows), eight chunks per load
// batch with the next batch in flight; the four waves' (max, sum, acc) then merge in a fixed order.
constexpr int CB_B = 8;  // chunks per load batch and wave
__global__ __launch_bounds__(256) void k_attn_combine(const float *__restrict__ part, float *__restrict__ out,
                                                      int hd, int n_chunks) {
    __shared__ float wm[AT_WAVES], wl[AT_WAVES], wo[AT_WAVES][64];
    const int i = blockIdx.x, lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int d = blockIdx.y * 64 + lane;
    const int dd = d < hd ? d : 0;
    const size_t stride = (size_t)hd + 2;
    const float *pp = part + (size_t)i * n_chunks * stride;
    const int nw = n_chunks > w ? (n_chunks - w + AT_WAVES - 1) / AT_WAVES : 0;  // this wave's chunks
    // clamped, always valid: past the wave's chunks its first one, or the row's last one if it has none
    auto chunk = [&](int j) { return j < nw ? w + AT_WAVES * j : min(w, n_chunks - 1); };
    // batch j: lane k < CB_B loads (m, l) of the wave's chunk j + k; every lane loads its dimension
    // of each of the CB_B chunks
    const int kl = lane < CB_B ? lane : 0;
    float a[CB_B], ml, ll;
    {
        const float *pc = pp + (size_t)chunk(kl) * stride;
        ml = pc[0];
        ll = pc[1];
#pragma unroll
        for (int k = 0; k < CB_B; ++k) a[k] = pp[(size_t)chunk(k) * stride + 2 + dd];
    }
    float M = -INFINITY, den = 0.0f, o = 0.0f;
    for (int j = 0; j < nw; j += CB_B) {
        float an[CB_B], mln, lln;
        {
            const float *pc = pp + (size_t)chunk(j + CB_B + kl) * stride;
            mln = pc[0];
            lln = pc[1];
#pragma unroll
            for (int k = 0; k < CB_B; ++k) an[k] = pp[(size_t)chunk(j + CB_B + k) * stride + 2 + dd];
        }
        float mc[CB_B], lc[CB_B];
        float bm = -INFINITY;
#pragma unroll
        for (int k = 0; k < CB_B; ++k) {
            mc[k] = readlane_f(ml, k);
            lc[k] = readlane_f(ll, k);
            if (j + k < nw) bm = fmaxf(bm, mc[k]);
        }
        const float Mn = fmaxf(M, bm);
        if (Mn != -INFINITY) {
            const float sc = M == -INFINITY ? 0.0f : expf(M - Mn);
            o *= sc;
            den *= sc;
#pragma unroll
            for (int k = 0; k < CB_B; ++k) {
                const float e = (j + k < nw && mc[k] != -INFINITY) ? expf(mc[k] - Mn) : 0.0f;
                o = fmaf(e, a[k], o);
                den = fmaf(e, lc[k], den);
            }
            M = Mn;
        }
#pragma unroll
        for (int k = 0; k < CB_B; ++k) a[k] = an[k];
        ml = mln;
        ll = lln;
    }
    if (lane == 0) {
        wm[w] = M;
        wl[w] = den;
    }
    wo[w][lane] = o;
    __syncthreads();
    if (w != 0 || d >= hd) return;
    const float Mx = fmaxf(fmaxf(wm[0], wm[1]), fmaxf(wm[2], wm[3]));
    float num = 0.0f, dsum = 0.0f;
#pragma unroll
    for (int u = 0; u < AT_WAVES; ++u) {
        const float e = wm[u] == -INFINITY ? 0.0f : expf(wm[u] - Mx);
        num = fmaf(e, wo[u][lane], num);
        dsum = fmaf(e, wl[u], dsum);
    }
    out[(size_t)i * hd + d] = num * (1.0f / dsum);
}

// The same merge for up to NW * CW chunks in one round of loads: wave w takes chunks w, w + NW, ..
// (at most CW), every value and lane k's (max, sum) of its k-th chunk loaded at once; the wave's
// maximum M_w, then o_w = sum_k e^(m_k - M_w) acc_k and l_w likewise in chunk order, and the NW
// waves' (M, l, o) merge in wave order as in k_attn_combine. Four waves of 32 chunks take up to
// 128 chunks, eight of 40 up to 320 (a global layer split into chunks of 64 keys at depth 16384).
template <int NW, int CW>
__global__ __launch_bounds__(NW * 64) void k_attn_merge(const float *__restrict__ part, float *__restrict__ out, int hd,
                                                        int n_chunks) {
    static_assert(CW <= 64, "one chunk's (max, sum) per lane");
    __shared__ float wm[NW], wl[NW], wo[NW][64];
    const int i = blockIdx.x, lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int d = blockIdx.y * 64 + lane;
    const int dd = d < hd ? d : 0;
    const size_t stride = (size_t)hd + 2;
    const float *pp = part + (size_t)i * n_chunks * stride;
    const int nw = n_chunks > w ? (n_chunks - w + NW - 1) / NW : 0;  // this wave's chunks
    // clamped, always valid: past the wave's chunks its first one, or the row's last one if it has none
    auto chunk = [&](int k) { return k < nw ? w + NW * k : min(w, n_chunks - 1); };
    float a[CW];
#pragma unroll
    for (int k = 0; k < CW; ++k) a[k] = pp[(size_t)chunk(k) * stride + 2 + dd];
    const int kl = lane < CW ? lane : 0;
    const float ml = pp[(size_t)chunk(kl) * stride], ll = pp[(size_t)chunk(kl) * stride + 1];
    const float mk = lane < nw ? ml : -INFINITY;
    float M = mk;
#pragma unroll
    for (int k = 0; k < CW; ++k) M = fmaxf(M, readlane_f(mk, k));
    const float e = mk == -INFINITY ? 0.0f : expf(mk - M);  // 0 past the wave's chunks and for empty ones
    float o = 0.0f, den = 0.0f;
#pragma unroll
    for (int k = 0; k < CW; ++k) {
        const float ek = readlane_f(e, k);
        o = fmaf(ek, a[k], o);
        den = fmaf(ek, readlane_f(ll, k), den);
    }
    if (lane == 0) {
        wm[w] = M;
        wl[w] = den;
    }
    wo[w][lane] = o;
    __syncthreads();
    if (w != 0 || d >= hd) return;
    float Mx = wm[0];
#pragma unroll
    for (int u = 1; u < NW; ++u) Mx = fmaxf(Mx, wm[u]);
    float num = 0.0f, dsum = 0.0f;
#pragma unroll
    for (int u = 0; u < NW; ++u) {
        const float eu = wm[u] == -INFINITY ? 0.0f : expf(wm[u] - Mx);
        num = fmaf(eu, wo[u][lane], num);
        dsum = fmaf(eu, wl[u], dsum);
    }
    out[(size_t)i * hd + d] = num * (1.0f / dsum);
}

// Q8_0 of the keys and values of tokens p0 .. p0 + n_tok - 1 into ring slots p % cap, bit for bit
// the CPU quantiser (runtime/src/ops.rs:95-105; the reference kernel is rvhip.hip:214-239): a thread
// per 4 elements, 8 per 32-value block, so that a wave loads 1 KB and stores each block's quants as
// eight dwords (one element per thread with byte stores took 5.96 us for 512 tokens of 8 heads of 256;
// the n_blk blocks of the keys come first, then the values').
__global__ __launch_bounds__(256) void k_kv_store(const float *__restrict__ k, const float *__restrict__ v,
                                                  uint8_t *__restrict__ kc, uint8_t *__restrict__ vc, int n_kv,
                                                  int hd, int p0, int cap, long n_blk) {
    const long i = (long)blockIdx.x * 32 + (threadIdx.x >> 3);
    const bool val = i >= n_blk, ok = i < 2 * n_blk;
    const long B = ok ? (val ? i - n_blk : i) : 0;  // (token, kv head, block)
    const int row = n_kv * (hd / QK);               // blocks per token
    const int t = (int)(B / row), b = (int)(B % row), e = threadIdx.x & 7;
    const F4u x = *(const F4u *)((val ? v : k) + B * QK + 4 * e);
    float m = 0.0f;
#pragma unroll
    for (int u = 0; u < 4; ++u) m = fmaxf(m, fabsf(x.v[u]));
    m = maxf_bits(m, dpp<0xb1>(__builtin_bit_cast(uint32_t, m)));
    m = maxf_bits(m, dpp<0x4e>(__builtin_bit_cast(uint32_t, m)));
    m = maxf_bits(m, dpp<0x141>(__builtin_bit_cast(uint32_t, m)));
    const float d = m / 127.0f;
    const float id = d != 0.0f ? 1.0f / d : 0.0f;
    uint32_t q = 0;
#pragma unroll
    for (int u = 0; u < 4; ++u) q |= (uint32_t)(uint8_t)(int8_t)sat_i8(roundf(x.v[u] * id)) << (8 * u);
    if (!ok) return;
    uint8_t *dst = (val ? vc : kc) + ((size_t)((p0 + t) % cap) * row + b) * Q8_BLOCK;
    *(Q8Word *)(dst + 2 + 4 * e) = Q8Word{q};
    if (e == 0) *(uint16_t *)dst = f2h_rne(d);
}

// The longest key range of a call (the last query's): it must fit the ring.
inline long attn_longest(int n_tok, int p0, int window) {
    const long last = (long)p0 + n_tok;
    return window > 0 && window < last ? (long)window : last;
}

// Heads per workgroup: the largest of 16, 8, 4, 2, 1 (8 for hd > 256) that divides the query heads
// of a kv head, halved while the smaller group's grid still fits the GPU in one round (workgroups
// resident per CU, from the runtime's occupancy for that kernel, times the CUs). Decode at depth
// has few tiles: a smaller head group spreads each tile's work over more CUs, which re-read its
// key and value rows from their XCD's L2; more workgroups than fit at once would only queue, as
// each is a serial chain of loads, scores, values and a merge.
template <int G, int DPL>
void launch_g(long wgs, const float *q, const uint8_t *kc, const uint8_t *vc, float *out, float *part, int n_tok,
              int n_head, int n_kv, int hd, int p0, int cap, int window, int n_chunks) {
    hipLaunchKernelGGL((k_attn_split<G, DPL>), dim3((unsigned)wgs), dim3(AT_WAVES * 64), 0, cur_stream(), q, kc, vc,
                       out, part, n_tok, n_head, n_kv, hd, p0, cap, window, n_chunks);
}

template <int G, int DPL>
long resident_wgs() {  // per GPU, for this kernel; cached per device
    static long cache[64] = {0};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
    if (cache[dev] == 0) {
        int per_cu = 0, cus = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_attn_split<G, DPL>, AT_WAVES * 64, 0) != hipSuccess ||
            hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || per_cu < 1 ||
            cus < 1)
            return 256;
        cache[dev] = (long)per_cu * cus;
    }
    return cache[dev];
}

template <int DPL>
long resident_for(int gt) {
    switch (gt) {
        case 16: return DPL == 4 ? resident_wgs<16, 4>() : 0;
        case 8: return resident_wgs<8, DPL>();
        case 4: return resident_wgs<4, DPL>();
        case 2: return resident_wgs<2, DPL>();
        default: return resident_wgs<1, DPL>();
    }
}

inline long attn_wgs(int n_tok, int n_head, int n_kv, int n_chunks, int gt) {
    const long tiles = (long)n_tok * n_kv * n_chunks;
    return (tiles + 7) / 8 * 8 * ((n_head / n_kv) / gt);  // see the workgroup mapping
}

template <int DPL>
int attn_group(int n_tok, int n_head, int n_kv, int n_chunks) {
    const int per_kv = n_head / n_kv;
    int gt = 1;
    for (int c = DPL == 8 ? 8 : 16; c > 1; c >>= 1)
        if (per_kv % c == 0) {
            gt = c;
            break;
        }
    while (gt > 1 && attn_wgs(n_tok, n_head, n_kv, n_chunks, gt / 2) <= resident_for<DPL>(gt / 2)) gt >>= 1;
    return gt;
}

// The streaming kernel's head group: every query head of a kv head, or groups of 16 when there are
// more (0 when it does not apply: another head dimension, or a count of heads 16 does not divide).
inline int stream_group(int n_head, int n_kv, int hd) {
    if (hd != 256 && hd != 512) return 0;
    const int per_kv = n_head / n_kv;
    return per_kv <= 16 ? per_kv : (per_kv % 16 == 0 ? 16 : 0);
}

int launch_stream(const float *q, const void *kc, const void *vc, float *out, float *part, int n_tok, int n_head,
                  int n_kv, int hd, int p0, int cap, int window, int n_chunks, int G, const float *kin,
                  const float *vin) {
    const long wgs = attn_wgs(n_tok, n_head, n_kv, n_chunks, G);
    RVM_CHECK(wgs <= 0x7fffffffL);
    // the rings are written only with kin / vin set (rvm_attn_decode, whose rings are writable)
    uint8_t *k8 = (uint8_t *)kc, *v8 = (uint8_t *)vc;
    if (hd == 512)
        hipLaunchKernelGGL(k_attn_stream<16>, dim3((unsigned)wgs), dim3(ST_WAVES * 64), 0, cur_stream(), q, k8, v8, out,
                           part, n_tok, n_head, n_kv, G, p0, cap, window, n_chunks, kin, vin);
    else
        hipLaunchKernelGGL(k_attn_stream<8>, dim3((unsigned)wgs), dim3(ST_WAVES * 64), 0, cur_stream(), q, k8, v8, out,
                           part, n_tok, n_head, n_kv, G, p0, cap, window, n_chunks, kin, vin);
    return launched();
}

// Several tokens of a head dimension of 2, 4, 8 or 16 blocks go through k_attn_prefill once the keys
// that the per-token kernels would read, tokens x kv heads x keys, are many: its workgroups have the
// longer start and merge. Measured, per-token kernel against this one (with the key/value store):
// hd 256, 2 tokens x 8 x 1024 keys 13.9 / 17.3 us, 24 x 8 x 300 21.3 / 23.9, 8 x 8 x 1024 25.1 / 22.1,
// 512 x 8 x 1024 745 / 48; hd 512, 2 x 2 x 3002 21.8 / 22.3, 8 x 2 x 3008 44.8 / 41.5, 500 x 2 x 4101
// 1244 / 247; hd 128, 2 x 4 x 512 13.8 / 14.1, 2 x 2 x 4002 25.0 / 18.0, 400 x 2 x 3400 1323 / 87; hd 64,
// 2 x 4 x 4002 23.4 / 14.0, 400 x 4 x 3400 1329 / 32. Four waves a workgroup for hd 128 (two workgroups
// per CU: 87 us against 98 with eight), eight for the others (hd 64: 32 against 42 with four).
//
// Several chunks shorten the per-token kernels' chains, so there the line lies higher (tokens x heads x keys in
// chunks, merged):
//  - hd 64 and 128: by rows x keys, as the per-token kernel computes every head apart, and further up where
//    its tiles of 64 keys are full: hd 128, 2 x 8 heads x 766 keys in 12 chunks 9.1 / 11.2, in 24 10.6 / 11.0,
//    16 x 4 x 376 in 6 10.7 / 11.5, 4 x 8 x 1024 in 16 10.8 / 11.1, 2 x 16 x 766 in 24 12.2 / 11.3; hd 64,
//    16 x 8 x 96 in 2 9.2 / 10.2, 2 x 8 x 1024 in 32 10.5 / 9.3;
//  - two tokens of at most two heads per kv head are 4 of 32 rows, and where they make more workgroups than CUs
//    the per-token kernel's shorter ones win: hd 128, 2 x 8 x 2251 in 36 12.4 / 14.4; hd 64 12.2 / 14.9 (but
//    hd 128, 2 x 8 x 4001 in 126 22.8 / 20.1);
//  - hd 256 and 512, four heads and more per kv head: k_attn_stream takes them at the price of one, and where its
//    grid just fits the CUs it is at its best: hd 256, 16 x 16 heads x 1021 keys in 4 chunks 21.8 / 25.3, x 1401
//    25.8 / 27.2 (in 8 chunks 30.8 / 22.8); hd 512, 16 x 8 x 1276 in 8 25.5 / 28.8 (in 16 33.7 / 25.1).
inline bool attn_prefill_ok(int n_tok, int n_head, int n_kv, int hd, int p0, int window, int n_chunks) {
    const long longest = attn_longest(n_tok, p0, window), keys = (long)n_tok * n_kv * longest;
    if (n_tok < 2 || (hd != 64 && hd != 128 && hd != 256 && hd != 512) ||
        keys < (hd > 256 ? 40000 : hd > 128 ? 64000 : 12000) || (long)n_tok * n_head > 0x7fffffffL - 64 ||
        (long)n_kv * (hd / QK * Q8_BLOCK) * PF_KEYS > 0x7fffffffL)
        return false;
    if (n_chunks == 1) return true;
    const int per_kv = n_head / n_kv, cus = device_cus();
    if (hd > 128) {
        const long wgs = (long)n_tok * n_kv * n_chunks;  // of k_attn_stream
        return per_kv < 4 || wgs > cus || wgs <= cus / 2 || keys >= (hd > 256 ? 60000 : 96000);
    }
    const long work = (long)n_tok * n_head * longest;
    const bool full = longest > 32L * n_chunks;  // chunks of more than half a tile of k_attn_split
    if (work < (hd == 64 ? (full ? 16500 : 12000) : (full ? 30000 : 16500))) return false;
    return n_tok > 2 || per_kv > 2 || (long)n_kv * n_chunks <= cus || work >= 50000;
}

template <int NBW, int TW, int WV>
int launch_prefill(const float *q, const uint8_t *kc, const uint8_t *vc, float *out, float *part, int n_tok, int n_head,
                   int n_kv, int p0, int cap, int window, int n_chunks) {
    const int tiles = grid_blocks((size_t)n_tok * (n_head / n_kv), PF_ROWS);
    RVM_CHECK((long)tiles * n_kv <= 0x7fffffffL / n_chunks);
    hipLaunchKernelGGL((k_attn_prefill<NBW, TW, WV>), dim3((unsigned)tiles * n_kv * n_chunks), dim3(WV * 64), 0,
                       cur_stream(), q, kc, vc, out, part, n_tok, n_head, n_kv, p0, cap, window, n_chunks, tiles);
    return launched();
}

int launch_attn(const float *q, const void *kc, const void *vc, float *out, float *part, int n_tok, int n_head,
                int n_kv, int hd, int p0, int cap, int window, int n_chunks) {
    if (attn_prefill_ok(n_tok, n_head, n_kv, hd, p0, window, n_chunks)) {
        const uint8_t *k8 = (const uint8_t *)kc, *v8 = (const uint8_t *)vc;
#define RVM_PREFILL_ARGS q, k8, v8, out, part, n_tok, n_head, n_kv, p0, cap, window, n_chunks
        if (hd == 512) return launch_prefill<4, 4, 8>(RVM_PREFILL_ARGS);
        if (hd == 256) return launch_prefill<4, 2, 8>(RVM_PREFILL_ARGS);
        if (hd == 128) return launch_prefill<4, 1, 4>(RVM_PREFILL_ARGS);
        return launch_prefill<2, 1, 8>(RVM_PREFILL_ARGS);
#undef RVM_PREFILL_ARGS
    }
    if (const int G = stream_group(n_head, n_kv, hd))
        return launch_stream(q, kc, vc, out, part, n_tok, n_head, n_kv, hd, p0, cap, window, n_chunks, G, nullptr,
                             nullptr);
    // heads per workgroup times dimensions per lane at most 64: the merge buffer's LDS
    const bool wide = hd > 256;
    const int gt = wide ? attn_group<8>(n_tok, n_head, n_kv, n_chunks) : attn_group<4>(n_tok, n_head, n_kv, n_chunks);
    const long wgs = attn_wgs(n_tok, n_head, n_kv, n_chunks, gt);
    RVM_CHECK(wgs <= 0x7fffffffL);
    const uint8_t *k8 = (const uint8_t *)kc, *v8 = (const uint8_t *)vc;
#define RVM_ATTN_ARGS wgs, q, k8, v8, out, part, n_tok, n_head, n_kv, hd, p0, cap, window, n_chunks
    if (wide) {
        switch (gt) {
            case 8: launch_g<8, 8>(RVM_ATTN_ARGS); break;
            case 4: launch_g<4, 8>(RVM_ATTN_ARGS); break;
            case 2: launch_g<2, 8>(RVM_ATTN_ARGS); break;
            default: launch_g<1, 8>(RVM_ATTN_ARGS); break;
        }
    } else {
        switch (gt) {
            case 16: launch_g<16, 4>(RVM_ATTN_ARGS); break;
            case 8: launch_g<8, 4>(RVM_ATTN_ARGS); break;
            case 4: launch_g<4, 4>(RVM_ATTN_ARGS); break;
            case 2: launch_g<2, 4>(RVM_ATTN_ARGS); break;
            default: launch_g<1, 4>(RVM_ATTN_ARGS); break;
        }
    }
#undef RVM_ATTN_ARGS
    return launched();
}

}  // namespace rvm

using namespace rvm;

extern "C" {

int rvh_kv_store(const float *k, const float *v, void *kc, void *vc, int n_tok, int n_kv, int hd, int p0, int cap) {
    RVM_CHECK(k && v && kc && vc && n_tok > 0 && n_kv > 0 && hd > 0 && hd % QK == 0 && p0 >= 0 && cap > 0);
    RVM_CHECK((long)n_tok * n_kv <= 0x7fffffffL);
    const long n_blk = (long)n_tok * n_kv * (hd / QK), wgs = (2 * n_blk + 31) / 32;
    RVM_CHECK(wgs <= 0x7fffffffL);
    hipLaunchKernelGGL(k_kv_store, dim3((unsigned)wgs), dim3(256), 0, cur_stream(), k, v, (uint8_t *)kc, (uint8_t *)vc,
                       n_kv, hd, p0, cap, n_blk);
    return launched();
}

int rvh_attn_split(const float *q, const void *kc, const void *vc, float *out, float *part, int n_tok, int n_head,
                   int n_kv, int hd, int p0, int cap, int window, int n_chunks) {
    RVM_CHECK(q && kc && vc && out && n_tok > 0 && n_kv > 0 && n_head > 0 && n_head % n_kv == 0 && hd > 0 &&
              hd % QK == 0 && hd <= AT_MAXHD && p0 >= 0 && cap > 0 && window >= 0 && n_chunks > 0 &&
              (n_chunks == 1 || part));
    RVM_CHECK(attn_longest(n_tok, p0, window) <= cap);
    return launch_attn(q, kc, vc, out, part, n_tok, n_head, n_kv, hd, p0, cap, window, n_chunks);
}

int rvh_attn_combine(const float *part, float *out, int rows, int hd, int n_chunks) {
    RVM_CHECK(part && out && rows > 0 && hd > 0 && n_chunks > 1);
    if (n_chunks > AT_WAVES * CB_B && n_chunks <= 4 * 32)  // more than one batch of k_attn_combine
        hipLaunchKernelGGL((k_attn_merge<4, 32>), dim3(rows, (hd + 63) / 64), dim3(4 * 64), 0, cur_stream(), part,
                           out, hd, n_chunks);
    else if (n_chunks > 4 * 32 && n_chunks <= 8 * 40)
        hipLaunchKernelGGL((k_attn_merge<8, 40>), dim3(rows, (hd + 63) / 64), dim3(8 * 64), 0, cur_stream(), part,
                           out, hd, n_chunks);
    else
        hipLaunchKernelGGL(k_attn_combine, dim3(rows, (hd + 63) / 64), dim3(AT_WAVES * 64), 0, cur_stream(), part,
                           out, hd, n_chunks);
    return launched();
}

int rvm_attn_decode(const float *q, const float *k, const float *v, void *kc, void *vc, float *out, float *part,
                    int n_head, int n_kv, int hd, int pos, int cap, int window, int n_chunks) {
    RVM_CHECK(q && k && v && kc && vc && out && n_kv > 0 && n_head > 0 && n_head % n_kv == 0 && hd > 0 &&
              hd % QK == 0 && hd <= AT_MAXHD && pos >= 0 && cap > 0 && window >= 0 && n_chunks > 0 &&
              (n_chunks == 1 || part));
    RVM_CHECK(attn_longest(1, pos, window) <= cap);
    const int G = stream_group(n_head, n_kv, hd);
    if (!G) {  // other shapes: the three reference operations in sequence
        if (int rc = rvh_kv_store(k, v, kc, vc, 1, n_kv, hd, pos, cap)) return rc;
        if (int rc = launch_attn(q, kc, vc, out, part, 1, n_head, n_kv, hd, pos, cap, window, n_chunks)) return rc;
    } else if (int rc = launch_stream(q, kc, vc, out, part, 1, n_head, n_kv, hd, pos, cap, window, n_chunks, G, k, v)) {
        return rc;
    }
    return n_chunks > 1 ? rvh_attn_combine(part, out, n_head, hd, n_chunks) : 0;
}

int rvh_attention(const float *q, const void *kc, const void *vc, float *out, float *scores, int n_tok, int n_head,
                  int n_kv, int hd, int p0, int cap, int window, int max_keys) {
    RVM_CHECK(q && kc && vc && out && scores && n_tok > 0 && n_kv > 0 && n_head > 0 && n_head % n_kv == 0 &&
              hd > 0 && hd % QK == 0 && hd <= AT_MAXHD && p0 >= 0 && cap > 0 && window >= 0);
    const long longest = attn_longest(n_tok, p0, window);
    RVM_CHECK(longest <= max_keys && longest <= cap);
    return launch_attn(q, kc, vc, out, nullptr, n_tok, n_head, n_kv, hd, p0, cap, window, 1);
}

}  // extern "C"
