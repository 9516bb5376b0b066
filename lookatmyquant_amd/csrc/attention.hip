// Causal grouped-query attention of the calibration forwards, fused: the score matrix never reaches memory.
//
// One workgroup per (sequence, head, block of 128 queries); its four waves take 32 queries each. The workgroup walks
// the key blocks of 64 up to its last query: each block's K and V rows (16 KB each) go straight from memory into LDS
// (global_load_lds, 16 bytes a lane, no registers), double-buffered, the next block's loads issued as soon as the
// current one is published (one barrier a block), so the four waves share one copy and no wave waits on a global
// load. Per block a wave forms S^T = K Q^T (two tiles of 32 keys x 32 queries: the head dim, 128, as eight 16-deep steps of
// v_mfma_f32_32x32x16_bf16 each, float32 sums) and masks it where the block reaches past its first query; then, half by
// half of 32 keys, it updates each query's running maximum and sum (the online softmax: exp2 with the scale and log2(e)
// folded into the scores), rounds the probabilities to bf16 and accumulates O^T += V^T P^T (128 x 32, float32); a wave
// past its own last query skips the half (whose block still arrives for the others). At the end O = O^T / sum, rounded
// to bf16 (nearest, ties to even).
//
// What bounds it: with two waves a SIMD the vector work of one runs under the matrix work of the other, 1,024 clocks a
// block, so the vector chain of a block is kept short: both halves' scores and maxima at once, no mask off the diagonal,
// the earlier sums rescaled only when some query's maximum has grown, the lanes of a query's keys combined by a swap of
// the wave's halves (LDS shuffles before), row pointers advanced a block at a time, and V's transposing reads issued
// before the softmax they are needed after. The results are those of 32 keys at a time, bit for bit: one softmax step
// for all 64 keys, its scale folded into a multiply-add, is another 7% faster, but a probability of the first half is
// then rounded to bf16 under a maximum it has not met (relative error against float64 of the 8-sequence case 2.01e-3
// -> 2.02e-3). 8 x 32 heads x 2,048: 657 -> 370-385 us (715-745 TFLOP/s); 32 sequences 2.59 -> 1.40 ms; one of 333
// tokens 14.9 -> 12.9 us.
// Workgroups go out pair by pair of sequence and key/value head, pairs spread over the XCDs, so that the query heads and
// blocks that read the same K and V run on one XCD together.
//
// Operand layouts (32x32x16 bf16 MFMA): A[m][k] has lane l holding m = l % 32 and k = 8 (l / 32) .. + 7; B[k][n]
// has lane l holding n = l % 32 and the same k; the result has lane l holding column l % 32 and rows
// 8 (v / 4) + 4 (l / 32) + v % 4 of register v. So S^T's result is P^T's B operand as it stands, with its k order
// (keys {0-3, 8-11} in lanes 0-31 and {4-7, 12-15} in lanes 32-63 for the first 16 keys, +16 for the second): the
// V^T operand takes the same order, as two transposing LDS reads (ds_read_b64_tr_b16: a 16-lane group reads a 4 x 16
// block, lane i receiving the four rows of column i) of four consecutive keys each. Q's fragments (B of S^T: eight
// consecutive head-dim values of one query) stay in registers; K's (A of S^T: eight consecutive head-dim values of
// one key) are 16-byte LDS reads. LDS rows are 256 bytes; K's 16-byte chunks are XOR-swizzled by (row & 15), so the
// 16 keys a fragment read serves at once touch 16 different chunks (all 64 banks once); V's by 4 (row & 3), so the
// 32 lanes a transposing read serves at once touch 16 different chunks of four rows. The loads place each chunk where
// the swizzle puts it (a lane fetches the chunk that belongs in its 16-byte slot).
#include "common.h"

typedef __bf16 lamq_at_bf16x8 __attribute__((ext_vector_type(8)));
typedef float lamq_at_f32x16 __attribute__((ext_vector_type(16)));

#define AT_GRID_X (1 << 22)
#define AT_D 128                        // head dim
#define AT_QW 32                        // queries per wave
#define AT_KB 32                        // keys per half block (one S^T tile)
#define AT_KB2 64                       // keys per block in LDS
#define AT_QB 128                       // queries per workgroup
#define AT_OPB (AT_KB2 * AT_D * 2)      // bytes of one operand's block (16 KB)

// byte offset of 16-byte chunk `chunk` (0..15) of row `row` in a V block, and in a K block
__device__ __forceinline__ uint32_t at_sw(int row, int chunk)
{
    return (uint32_t)(row * (AT_D * 2) + ((chunk ^ (4 * (row & 3))) << 4));
}
__device__ __forceinline__ uint32_t at_ksw(int row, int chunk)
{
    return (uint32_t)(row * (AT_D * 2) + ((chunk ^ (row & 15)) << 4));
}

typedef short lamq_at_s4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) lamq_at_s4 lamq_at_lds_s4;

// the larger of this lane's value and lane ^ 32's (one swap of the wave's halves, no LDS)
__device__ __forceinline__ float at_max32(float v)
{
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float at_sum32(float v)
{
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void attention_causal_kernel(
    const uint16_t* __restrict__ Q, int64_t sqb, int64_t sqh, int64_t sqt, const uint16_t* __restrict__ K,
    int64_t skb, int64_t skh, int64_t skt, const uint16_t* __restrict__ V, int64_t svb, int64_t svh, int64_t svt,
    uint16_t* __restrict__ O, int64_t sob, int64_t soh, int64_t sot, int rep, int Hkv, int pairs, int T, float scale_log2)
{
    __shared__ __align__(16) uint8_t lds[2][2][AT_OPB];  // [buffer][K, V]
    const int nqb = (T + AT_QB - 1) / AT_QB;
    // workgroup -> (pair of sequence and key/value head, query head of the pair, query block)
    int pair, rem;
    {
        const int id = (int)(blockIdx.y * gridDim.x + blockIdx.x), per = nqb * rep;
        if ((unsigned)id >= (unsigned)pairs * (unsigned)per) return;  // past the last (the grid's last row)
        if (pairs % LAMQ_XCDS == 0) {
            const int y = id / LAMQ_XCDS;
            pair = y / per * LAMQ_XCDS + id % LAMQ_XCDS;
            rem = y % per;
        } else {
            pair = id / per;
            rem = id % per;
        }
    }
    const int qb = nqb - 1 - rem / rep;  // the longest query blocks first
    const int b = pair / Hkv, hk = pair % Hkv, h = hk * rep + rem % rep;
    const int wave = (int)(threadIdx.x >> 6), lane = (int)(threadIdx.x & 63);
    const int wv = __builtin_amdgcn_readfirstlane(wave);
    const int q0 = qb * AT_QB + AT_QW * wv;
    const int li = lane & 31, hi = lane >> 5, g = lane >> 4, i16 = lane & 15;
    const uint16_t* Qp = Q + b * sqb + (int64_t)h * sqh;
    const uint16_t* Kp = K + b * skb + (int64_t)hk * skh;
    const uint16_t* Vp = V + b * svb + (int64_t)hk * svh;
    const uint32_t base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)lds;
    // every wave takes part in the loads and barriers up to the workgroup's last query; a wave's own work ends at its
    // last query (none for a wave wholly past T)
    const int wg_last = (qb * AT_QB + AT_QB < T ? qb * AT_QB + AT_QB : T) - 1;
    const int nblk = wg_last / AT_KB2 + 1;
    const int my_last = q0 < T ? (q0 + AT_QW < T ? q0 + AT_QW : T) - 1 : -1;
    // block kb's rows into buffer kb & 1: instruction i (four a wave and operand) covers rows 4i .. 4i + 3, lane l row
    // 4i + l / 16, slot l % 16. The row pointers advance a block at a time; in a block that reaches past T the rows there
    // read row T - 1 (finite values that meet zero probabilities)
    const int lrow = 16 * wv + (lane >> 4), slot = lane & 15;
    const uint16_t* kp[4];
    const uint16_t* vp[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int row = lrow + 4 * q;
        kp[q] = Kp + row * skt + 8 * (slot ^ (row & 15));
        vp[q] = Vp + row * svt + 8 * (slot ^ (4 * (row & 3)));
    }
    auto load_block = [&](int kb) {
        const uint32_t kbuf = base + (uint32_t)((kb & 1) * 2 * AT_OPB), vbuf = kbuf + AT_OPB;
        const int over = kb * AT_KB2 + AT_KB2 - T;  // rows past T
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int i = 4 * wv + q;
            const uint16_t *ka = kp[q], *va = vp[q];
            if (over > 0) {  // uniform
                const int back = lrow + 4 * q - (AT_KB2 - 1 - over);  // this row's distance past row T - 1
                if (back > 0) {
                    ka -= back * skt;
                    va -= back * svt;
                }
            }
            load_lds16(ka, kbuf + (uint32_t)(i * 1024));
            load_lds16(va, vbuf + (uint32_t)(i * 1024));
            kp[q] += AT_KB2 * skt;
            vp[q] += AT_KB2 * svt;
        }
    };
    load_block(0);
    const int myq = q0 + li;  // this lane's query (past T: computed, not stored)
    const int qrow = myq < T ? myq : T - 1;
    lamq_at_bf16x8 qf[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) qf[j] = *reinterpret_cast<const lamq_at_bf16x8*>(Qp + qrow * sqt + 16 * j + 8 * hi);
    // the Q fragments as operands of an empty asm: the compiler waits for their loads here, before the loop. The
    // loop's own waits are asm, invisible to it, so without this it would wait on the Q loads inside the loop, where
    // its counts would cover the next block's loads as well and stall their prefetch
    asm volatile("" : "+v"(qf[0]), "+v"(qf[1]), "+v"(qf[2]), "+v"(qf[3]), "+v"(qf[4]), "+v"(qf[5]), "+v"(qf[6]),
                 "+v"(qf[7]));
    lamq_at_f32x16 o[4];
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int v = 0; v < 16; ++v) o[t][v] = 0.0f;
    float mrun = -__builtin_inff(), lrun = 0.0f;  // each query's maximum (of the scaled scores) and sum
    for (int kb = 0; kb < nblk; ++kb) {
        wait_vm<0>();     // this wave's loads of block kb have landed
        __syncthreads();  // everyone's; the other buffer (block kb - 1) is free
        if (kb + 1 < nblk) load_block(kb + 1);
        const int k0 = kb * AT_KB2;
        if (k0 > my_last) continue;  // uniform: this wave's queries end before these keys
        const uint8_t* kl = lds[kb & 1][0];
        const uint32_t vbase = base + (uint32_t)(((kb & 1) * 2 + 1) * AT_OPB);
        // S^T, two tiles of 32 keys: K fragments (A) of key 32 hf + li, head dims 16 j + 8 hi .. + 7 (chunk 2 j + hi)
        lamq_at_f32x16 s[2];
#pragma unroll
        for (int hf = 0; hf < 2; ++hf)
#pragma unroll
            for (int v = 0; v < 16; ++v) s[hf][v] = 0.0f;
#pragma unroll
        for (int j = 0; j < 8; ++j)
#pragma unroll
            for (int hf = 0; hf < 2; ++hf) {
                const lamq_at_bf16x8 kf =
                    *reinterpret_cast<const lamq_at_bf16x8*>(kl + at_ksw(AT_KB * hf + li, 2 * j + hi));
                s[hf] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, qf[j], s[hf], 0, 0, 0);
            }
        // V fragments, sixteen transposing reads a half, under the softmax. Lane: head dim 32 t + li; keys 16 mi + 4 hi +
        // {0..3} and + 8 of the half (the P^T order); the group's lane i16 points at row 32 hf + 16 mi + 4 hi + i16 / 4,
        // columns 32 t + 16 (g & 1) + 4 (i16 % 4) .. + 3
        lamq_at_s4 vf[2][4][2][2];
#pragma unroll
        for (int hf = 0; hf < 2; ++hf)
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int mi = 0; mi < 2; ++mi) {
                    const int row = AT_KB * hf + 16 * mi + 4 * hi + (i16 >> 2);
                    const int col = 32 * t + 16 * (g & 1) + 4 * (i16 & 3);
                    const uint32_t a0 = vbase + at_sw(row, col >> 3) + 8 * ((col >> 2) & 1);
                    const uint32_t a1 = vbase + at_sw(row + 8, col >> 3) + 8 * ((col >> 2) & 1);
                    vf[hf][t][mi][0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lamq_at_lds_s4*)(uintptr_t)a0);
                    vf[hf][t][mi][1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lamq_at_lds_s4*)(uintptr_t)a1);
                }
        // the causal mask, only where the block reaches past the wave's first query (a key past T is past every query
        // below T too)
        if (k0 + AT_KB2 - 1 > q0) {
#pragma unroll
            for (int hf = 0; hf < 2; ++hf)
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    const int key = k0 + AT_KB * hf + 8 * (v >> 2) + 4 * hi + (v & 3);
                    s[hf][v] = key <= myq ? s[hf][v] : -__builtin_inff();
                }
        }
        // the running maximum after each half's 32 keys (finite from the first half on: key 0 is never masked). The scale
        // is positive and its product rounded monotonically, so the scaled maximum is the maximum of the scaled scores
        float m[2];
#pragma unroll
        for (int hf = 0; hf < 2; ++hf) {
            float mx = s[hf][0];
#pragma unroll
            for (int v = 1; v < 16; ++v) mx = fmaxf(mx, s[hf][v]);
            m[hf] = fmaxf(hf == 0 ? mrun : m[0], at_max32(mx) * scale_log2);
        }
#pragma unroll
        for (int hf = 0; hf < 2; ++hf)
            // uniform; a half past the wave's last query has no part in the sums
            if (hf == 0 || k0 + AT_KB <= my_last) {
                lamq_at_bf16x8 pf[2];
                float ps = 0.0f;
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    const float x = s[hf][v] * scale_log2;
                    const float p = __builtin_amdgcn_exp2f(x - m[hf]);  // masked: exp2(-inf) = 0
                    ps += p;
                    pf[v >> 3][v & 7] = (__bf16)p;
                }
                // the sums are rescaled only in halves where some query's maximum grows (elsewhere by exactly 1)
                if (__builtin_amdgcn_ballot_w64(m[hf] > mrun)) {
                    const float alpha = __builtin_amdgcn_exp2f(mrun - m[hf]);  // 0 on the first half
                    lrun *= alpha;
                    mrun = m[hf];
#pragma unroll
                    for (int t = 0; t < 4; ++t)
#pragma unroll
                        for (int v = 0; v < 16; ++v) o[t][v] *= alpha;
                }
                lrun += at_sum32(ps);
#pragma unroll
                for (int mi = 0; mi < 2; ++mi)
#pragma unroll
                    for (int t = 0; t < 4; ++t) {
                        const short __attribute__((ext_vector_type(8))) w =
                            __builtin_shufflevector(vf[hf][t][mi][0], vf[hf][t][mi][1], 0, 1, 2, 3, 4, 5, 6, 7);
                        o[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(lamq_at_bf16x8, w), pf[mi],
                                                                       o[t], 0, 0, 0);
                    }
            }
        // the next iteration's barrier comes after every wave's reads of this buffer (their results are used above)
    }
    if (myq >= T) return;
    const float inv = 1.0f / lrun;
    uint16_t* Op = O + b * sob + (int64_t)h * soh + (int64_t)myq * sot;
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            // registers 4 r .. 4 r + 3: head dims 32 t + 8 r + 4 hi + {0..3}
            uint32_t w2[2];
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const __bf16 x0 = (__bf16)(o[t][4 * r + 2 * e] * inv), x1 = (__bf16)(o[t][4 * r + 2 * e + 1] * inv);
                w2[e] = (uint32_t)__builtin_bit_cast(uint16_t, x0) | ((uint32_t)__builtin_bit_cast(uint16_t, x1) << 16);
            }
            *reinterpret_cast<uint2*>(Op + 32 * t + 8 * r + 4 * hi) = make_uint2(w2[0], w2[1]);
        }
}

// out[b, t, h, :] = softmax(q[b, h, t, :] k[b, h / rep, :t + 1, :]^T * scale) v[b, h / rep, :t + 1, :], bf16 in and out;
// every tensor's head dim (128) contiguous, the other strides in elements.
extern "C" int lamq_attention_causal_bf16(const uint16_t* q, int64_t sqb, int64_t sqh, int64_t sqt, const uint16_t* k,
                                          int64_t skb, int64_t skh, int64_t skt, const uint16_t* v, int64_t svb,
                                          int64_t svh, int64_t svt, uint16_t* out, int64_t sob, int64_t soh,
                                          int64_t sot, int64_t B, int64_t H, int64_t Hkv, int64_t T, int64_t D,
                                          float scale, void* stream)
{
    if (!q || !k || !v || !out || B < 0 || H < 1 || Hkv < 1 || T < 0 || H % Hkv != 0) return LAMQ_EINVAL;
    if (D != AT_D) return LAMQ_EUNSUP;
    if (!(scale > 0.0f) || !(scale < 3.0e38f)) return LAMQ_EINVAL;
    const int64_t strides[12] = {sqb, sqh, sqt, skb, skh, skt, svb, svh, svt, sob, soh, sot};
    for (int64_t s : strides)
        if (s < 0 || s % 8 != 0) return LAMQ_EINVAL;  // 16-byte rows of eight bf16
    if (((uintptr_t)q % 16) || ((uintptr_t)k % 16) || ((uintptr_t)v % 16) || ((uintptr_t)out % 8)) return LAMQ_EINVAL;
    if (B == 0 || T == 0) return LAMQ_OK;
    if (B > 65535 || H > 65535 || T > 0x7fffff) return LAMQ_EUNSUP;
    if (cdiv(T, AT_QB) * H * B > 0x7fffffff) return LAMQ_EUNSUP;
    // a grid's work items along x must stay below 2^32, so past 2^22 workgroups they go out in rows
    const int64_t wgs = cdiv(T, AT_QB) * H * B, gx = wgs < AT_GRID_X ? wgs : AT_GRID_X;
    const dim3 grid((unsigned)gx, (unsigned)cdiv(wgs, gx));
    hipLaunchKernelGGL(attention_causal_kernel, grid, dim3(256), 0, as_stream(stream), q, sqb, sqh, sqt, k, skb, skh, skt,
                       v, svb, svh, svt, out, sob, soh, sot, (int)(H / Hkv), (int)Hkv, (int)(B * Hkv), (int)T,
                       scale * 1.4426950408889634f);
    LAMQ_LAUNCH_CHECK();
    return LAMQ_OK;
}
