// Prefill MUL_MAT (many tokens) on the int8 matrix cores of MI355X with ggml's exact block integers.
//
// Role of ameva_mmq.comp:55-163 / ameva_mmqb.comp:11-16, 54-157 (reference, enc_mul_mat_mmq ggml-ameva.cpp:2540-2647):
// dst[m][n] = sum over the blocks of row n of the f32 epilogue of one exact integer per block, as ggml's
// vec_dot_q4_0_q8_0 / q8_0_q8_0 / q4_K_q8_K compute it on the CPU:
//   Q4_0 / Q8_0 (32-blocks):  S = sum_k w_k q_k (w = q - 8 or q),           dst += S * d_a * d_w
//   Q4_K (256-blocks of 8 units of 32, 6-bit scales sc_u and mins m_u):
//                             I1 = sum_u sc_u sum_k q_k a_k, I2 = sum_u m_u sum_k a_k,
//                             dst += d_a * (d * I1 - dmin * I2)
// One v_mfma_i32_32x32x32_i8 is one 32-block (or one Q4_K unit) of a 32 x 32 tile, so S comes out of the matrix core
// as an int32, exact. The per-block epilogue is VALU work beside the matrix core and bounds these kernels: Q4_0 / Q8_0 take
// two operations per output and block (convert, fma), Q4_K one integer multiply-add per unit (I1 += sc_u S_u) and four
// per super-block (I2 is one f16 MFMA of the units' mins against the activation sums per 16, exact in f32).
// The inputs are the plain activation layouts (int8 q with {f32 d, i32 sum} per 32, or Q8_K's f32 d per 256 and i32
// sums per 16): no f16 copies are read.
//
// MFMA operands: A = tokens, B = weight rows; lane l supplies token (row of A) / weight row (column of B) l % 32 and the 16
// bytes 16 (l / 32) .. + 15 of the 32-block (any assignment of k to byte slots works as long as A and B share it); the
// result D of lane l holds weight row l % 32 and tokens 8 (r / 4) + 4 (l / 32) + r % 4, r = 0..15.
// The grid is one dimension, mapped so that the workgroups sharing a weight tile (its token tiles) are dispatched to
// the same XCD, one after another, and with a split of k each k range goes to its own group of XCDs (range z to
// XCDs 8 z / n_z ..): MI355X hands workgroup i to XCD i % 8, and each XCD has its own L2, so an XCD reads the weight
// rows of its tiles once and only its k range of the activation (on the 4096 x 14336 down shape at M = 512 with k
// split in two this cut the L2 -> memory reads from 118 to 70 MB per launch, at the same time).
#include "amv_common.h"

#include <algorithm>

typedef int qg_v4i __attribute__((ext_vector_type(4)));
typedef int qg_v16i __attribute__((ext_vector_type(16)));
typedef _Float16 qg_h8 __attribute__((ext_vector_type(8)));
typedef float qg_f16v __attribute__((ext_vector_type(16)));

// byte-wise n - 8 of nibbles n in 0..15 (no carry crosses a byte: n + 0x78 <= 0x87)
__device__ __forceinline__ uint32_t qg_m8(uint32_t v) { return (v + 0x78787878u) ^ 0x80808080u; }

// ---------------------------------------------------------------------------------------------------------------
// Q4_0 / Q8_0 x Q8_0. Bytes go from memory to LDS without registers (buffer_load .. lds), one step of four blocks (128 k)
// ahead; Q4_0 weights stay packed there and a lane unpacks its operand bytes (n - 8 per byte) for both its token tiles.
// Per wave 64 tokens x 32 rows: WM x WN waves on BM = 64 WM tokens x BN = 32 WN rows, KG such groups in a workgroup on
// consecutive parts of k, their sums added at the end: where the tiles alone leave at most one workgroup per CU, a group by
// itself waits for its loads most of the time. The registers stay within 128, so four waves share a SIMD.
// Epilogue of a block: the scale products d_a d_w of both token tiles are one outer product on the matrix core
// (v_mfma_f32_32x32x1_2b_f32: each one f32 product), which leaves the conversion and the fma.
// LDS rows are unpadded (the loads write them as they come): the 16-byte pieces of a row are exchanged by an XOR with the
// row index on the memory side, so that the fragment reads of 16 consecutive rows hit all banks once.
// ---------------------------------------------------------------------------------------------------------------
typedef __attribute__((address_space(3))) void qg_lds;
#define QG_RSRC(p, bytes) __builtin_amdgcn_make_buffer_rsrc((void*)(p), 0, (uint32_t)(bytes), 0x00027000)
// wait for every vector memory load (the other counters are left alone)
#define QG_WAIT_LOADS() __builtin_amdgcn_s_waitcnt(0x0f70)

// The end of a product: the KG groups' sums joined in the first group, in order of k, through the first A buffers (gA: KG
// x BM * 8 pieces, free), 8 registers of a thread at a time, then stored. A lane holds weight row n and tokens
// m + 32 i + 8 (r / 4) + r % 4: for each r the 32 lanes of a half store 32 consecutive floats of one token row.
template <bool SUMS, int BM, int NT, int KG, bool ADD>
__device__ __forceinline__ void qg_finish(qg_f16v (&acc)[2], uint4 (*gA)[BM * 8], int kg, int t, int n, int m, int M, int N,
                                          float* __restrict__ dst, int64_t ldd, const float* add) {
    if constexpr (SUMS) return;
    if constexpr (KG > 1) {
        constexpr int PER = BM * 8 * 4 / NT;
        float* const red = reinterpret_cast<float*>(gA[kg]);
#pragma unroll
        for (int q = 0; q < 32 / PER; ++q) {
            __syncthreads();
            if (kg)
#pragma unroll
                for (int r = 0; r < PER; ++r) red[r * NT + t] = acc[(q * PER + r) / 16][(q * PER + r) % 16];
            __syncthreads();
            if (!kg)
#pragma unroll
                for (int g = 1; g < KG; ++g)
#pragma unroll
                    for (int r = 0; r < PER; ++r)
                        acc[(q * PER + r) / 16][(q * PER + r) % 16] += reinterpret_cast<const float*>(gA[g])[r * NT + t];
        }
        if (kg) return;
    }
    if (n >= N) return;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int mm = m + 32 * i + 8 * (r >> 2) + (r & 3);
            if (mm < M) {
                const size_t o = (size_t)mm * ldd + n;
                if constexpr (ADD) dst[o] = acc[i][r] + add[o];
                else dst[o] = acc[i][r];
            }
        }
}

template <int WT, bool SUMS, int WM, int WN, int KG, bool ADD = false>
__global__ __launch_bounds__(64 * WM * WN * KG) __attribute__((amdgpu_waves_per_eu(4))) void k_qgemm(
    const uint8_t* __restrict__ wq, const uint16_t* __restrict__ wd, int N, int nb, const int8_t* __restrict__ aq,
    const int2* __restrict__ am, int M, float* __restrict__ dst, int64_t ldd, const float* add,
    int32_t* __restrict__ sums, int kb_per, int64_t zstride, int n_tw, int n_tt, int n_z) {
    constexpr int BN = 32 * WN, BM = 64 * WM, NT = 64 * WM * WN;
    constexpr bool Q4 = WT == AMV_T_Q4_0;
    constexpr int WB = Q4 ? 16 : 32, WP = 4 * WB / 16;            // bytes of a weight block, 16-byte pieces of a step's row
    constexpr int RA = BM * 8 / NT, RW = BN * WP / NT;            // rounds of the threads over a step's pieces
    constexpr int RDA = BM * 4 / NT, RDW = BN * 4 / NT;           // and over its scales
    // the buffers of even and odd steps are variables of their own: reads of one do not wait for the loads into the other
    __shared__ __align__(16) uint4 gAa[KG][BM * 8], gAb[KG][BM * 8], gWa[KG][BN * WP], gWb[KG][BN * WP];
    __shared__ __align__(16) float gDa[KG][2][4 * BM], gDw[KG][2][4 * BN];
    const int t = threadIdx.x & (NT - 1), lane = t & 63, c32 = lane & 31, h = lane >> 5;
    const int kg = KG == 1 ? 0 : __builtin_amdgcn_readfirstlane((int)threadIdx.x / NT);
    uint4 *const sAa = gAa[kg], *const sAb = gAb[kg], *const sWa = gWa[kg], *const sWb = gWb[kg];
    const int wv = __builtin_amdgcn_readfirstlane(t >> 6), wm = wv / WN, wn = wv % WN;
    // tile index: token tile fastest, then the split of k, then the weight tile
    const int T = amv_xcd_tile(blockIdx.x, n_tw * n_z * n_tt);
    const int tt = T % n_tt, tw = (T / n_tt) % n_tw, z = T / (n_tt * n_tw);
    const int n0 = tw * BN, m0 = tt * BM;
    const int K = nb * 32;
    // the split's blocks, dealt to the KG groups of waves in runs of steps
    const int z0 = z * kb_per, z_end = min(nb, z0 + kb_per), nsteps = ((z_end - z0 + 3) / 4 + KG - 1) / KG;
    const int b0 = z0 + 4 * nsteps * kg, b_end = min(z_end, b0 + 4 * nsteps);
    dst += (size_t)z * zstride;

    // Rows past N, tokens past M and, behind the last of them, blocks past the end (a partial last step, the prefetch after
    // it, groups without blocks) read as zero. A buffer's range check leaves out the scalar offset, so each step has a
    // buffer that begins at its first block. Behind any other row blocks past the end are the next row's, and unused.
    const int mr = min(BM, M - m0), nr = min(BN, N - n0);
    const int8_t* const pa = aq + (size_t)m0 * K;
    const uint8_t* const pw = wq + (size_t)n0 * nb * WB;
    const __amdgpu_buffer_rsrc_t rm = QG_RSRC(am + (size_t)m0 * nb, (uint32_t)(mr * nb) * 8u);
    const uint32_t oa = (uint32_t)(t >> 3) * K + 16 * ((t & 7) ^ ((t >> 4) & 7));
    const uint32_t ow = Q4 ? (uint32_t)(t >> 2) * (nb * 16) + 16 * ((t & 3) ^ ((t >> 4) & 3))
                           : (uint32_t)(t >> 3) * (nb * 32) + 16 * ((t & 7) ^ ((t >> 4) & 7));
    const auto load = [&](uint4* sA, uint4* sW, int b) {
        const int bc = min(b, nb);
        const __amdgpu_buffer_rsrc_t ra = QG_RSRC(pa + 32 * bc, (uint32_t)mr * K - 32u * bc);
        const __amdgpu_buffer_rsrc_t rw = QG_RSRC(pw + WB * bc, (uint32_t)nr * (nb * WB) - (uint32_t)WB * bc);
#pragma unroll
        for (int i = 0; i < RA; ++i)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (qg_lds*)(sA + NT * i + 64 * wv), 16,
                                                     oa + (uint32_t)(NT / 8 * i) * K, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < RW; ++i)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rw, (qg_lds*)(sW + NT * i + 64 * wv), 16,
                                                     ow + (uint32_t)(NT / WP * i) * (nb * WB), 0, 0, 0);
    };
    // scales, through registers: token x / 4 (row x / 4) of the block x % 4 of the step; 0 past the group's blocks
    float da[RDA];
    uint32_t dw[RDW];
    const auto load_s = [&](int b) {
#pragma unroll
        for (int i = 0; i < RDA; ++i) {
            const int x = t + NT * i, bb = b + (x & 3);
            da[i] = __int_as_float(
                __builtin_amdgcn_raw_buffer_load_b32(rm, ((uint32_t)(x >> 2) * nb + (bb < b_end ? bb : 0)) * 8u, 0, 0));
        }
#pragma unroll
        for (int i = 0; i < RDW; ++i) {
            const int x = t + NT * i, bb = min(b + (x & 3), z_end - 1), row = min(n0 + (x >> 2), N - 1);
            dw[i] = wd[Q4 ? amv_q4_0_didx(row, bb, nb, N) : (size_t)row * nb + bb];
        }
    };
    const auto store_s = [&](int b, int buf) {
#pragma unroll
        for (int i = 0; i < RDA; ++i) {
            const int x = t + NT * i;
            gDa[kg][buf][(x & 3) * BM + (x >> 2)] = b + (x & 3) < b_end ? da[i] : 0.0f;
        }
#pragma unroll
        for (int i = 0; i < RDW; ++i) {
            const int x = t + NT * i;
            gDw[kg][buf][(x & 3) * BN + (x >> 2)] = b + (x & 3) < b_end ? amv_h2f((uint16_t)dw[i]) : 0.0f;
        }
    };

    qg_f16v acc[2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][r] = 0.0f;
    const int ar = 64 * wm + c32, wr = 32 * wn + c32;
    const int ax = (c32 >> 1) & 7, wx = Q4 ? (c32 >> 2) & 3 : ax;  // the rows' XOR (64 wm, 32 i, 32 wn do not change them)
    const auto compute = [&](const uint4* sA, const uint4* sW, int b, int buf) {
#pragma unroll
        for (int bl = 0; bl < 4; ++bl) {
            typedef float f32v __attribute__((ext_vector_type(32)));
            f32v o;
            if constexpr (!SUMS) {
                const f32v zero = {};
                o = __builtin_amdgcn_mfma_f32_32x32x1f32(gDa[kg][buf][bl * BM + 64 * wm + lane], gDw[kg][buf][bl * BN + wr],
                                                         zero, 0, 0, 0);
            }
            qg_v4i B;
            if constexpr (Q4) {  // element e < 16: low nibble of byte e (lane half 0); 16 + e: its high nibble (half 1)
                const uint4 x = sW[wr * 4 + (bl ^ wx)];
                const int s = 4 * h;
                B = qg_v4i{(int)qg_m8((x.x >> s) & 0x0F0F0F0Fu), (int)qg_m8((x.y >> s) & 0x0F0F0F0Fu),
                           (int)qg_m8((x.z >> s) & 0x0F0F0F0Fu), (int)qg_m8((x.w >> s) & 0x0F0F0F0Fu)};
            } else {
                const uint4 x = sW[wr * 8 + ((2 * bl + h) ^ wx)];
                B = qg_v4i{(int)x.x, (int)x.y, (int)x.z, (int)x.w};
            }
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const uint4 a = sA[(ar + 32 * i) * 8 + ((2 * bl + h) ^ ax)];
                const qg_v16i zero = {};
                const qg_v16i C = __builtin_amdgcn_mfma_i32_32x32x32_i8(
                    qg_v4i{(int)a.x, (int)a.y, (int)a.z, (int)a.w}, B, zero, 0, 0, 0);
                if constexpr (SUMS) {
                    const int n = n0 + wr;
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        const int m = m0 + 64 * wm + 32 * i + 8 * (r >> 2) + 4 * h + (r & 3);
                        if (b + bl < b_end && m < M && n < N) sums[((size_t)m * N + n) * nb + b + bl] = C[r];
                    }
                } else {
#pragma unroll
                    for (int r = 0; r < 16; ++r) acc[i][r] = fmaf((float)C[r], o[16 * i + r], acc[i][r]);
                }
            }
            // one block's results at a time (more do not fit the registers), added up here (the compiler would move the
            // additions behind the next barrier and keep the results until then)
            asm volatile("" : "+v"(acc[0]), "+v"(acc[1]));
            __builtin_amdgcn_sched_barrier(0);
        }
    };

    load(sAa, sWa, b0);
    load_s(b0);
    store_s(b0, 0);
    QG_WAIT_LOADS();
    __syncthreads();
    for (int s = 0;; s += 2) {
        load(sAb, sWb, b0 + 4 * (s + 1));
        load_s(b0 + 4 * (s + 1));
        if (b0 + 4 * s < b_end) compute(sAa, sWa, b0 + 4 * s, 0);
        if (s + 1 >= nsteps) break;
        store_s(b0 + 4 * (s + 1), 1);
        QG_WAIT_LOADS();
        __syncthreads();
        load(sAa, sWa, b0 + 4 * (s + 2));
        load_s(b0 + 4 * (s + 2));
        if (b0 + 4 * (s + 1) < b_end) compute(sAb, sWb, b0 + 4 * (s + 1), 1);
        if (s + 2 >= nsteps) break;
        store_s(b0 + 4 * (s + 2), 0);
        QG_WAIT_LOADS();
        __syncthreads();
    }
    QG_WAIT_LOADS();  // the last step's prefetch may still write LDS
    qg_finish<SUMS, BM, NT, KG, ADD>(acc, gAa, kg, t, n0 + wr, m0 + 64 * wm + 4 * h, M, N, dst, ldd, add);
}

// ---------------------------------------------------------------------------------------------------------------
// Q4_K x Q8_K. All operands go from memory to LDS without registers (buffer_load .. lds), one step ahead, and the
// weights stay packed there: the 16 bytes a lane reads of a 32-byte chunk are its operand bytes of two units (low and
// high nibbles), unpacked in 12 operations for both token tiles. Waves, groups and LDS rows as k_qgemm above: with the loads staged
// through registers and two waves of 64 x 64 on a SIMD, half the cycles went by with no instruction issued.
// Step = half a super-block (128 k).
// Per super-block: the 16-byte heads go to LDS with the first half; every lane decodes its row's 8 scales and mins from
// the head (bytes, 8 operations). The activation sums per 16 (f16) and d_a are staged through registers.
// ---------------------------------------------------------------------------------------------------------------
__device__ __forceinline__ uint32_t qg_h2(int a, int b) {
    return (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)(float)a) |
           ((uint32_t)__builtin_bit_cast(uint16_t, (_Float16)(float)b) << 16);
}

template <bool SUMS, int WM, int WN, int KG, bool ADD = false>
__global__ __launch_bounds__(64 * WM * WN * KG) __attribute__((amdgpu_waves_per_eu(4))) void k_qgemm_q4k(
    const uint4* __restrict__ wq, const uint4* __restrict__ wh, int N, int nsb, const int8_t* __restrict__ aq,
    const float* __restrict__ ad, const int32_t* __restrict__ as16, int M, float* __restrict__ dst, int64_t ldd,
    const float* add, int32_t* __restrict__ sums, int sb_per, int64_t zstride, int n_tw, int n_tt, int n_z) {
    constexpr int BN = 32 * WN, BM = 64 * WM, NT = 64 * WM * WN;
    constexpr int RA = BM * 8 / NT, RW = BN * 4 / NT, RS = BM * 4 / NT;  // rounds of the threads over a step's pieces
    // the buffers of the two halves are variables of their own: reads of one do not wait for the loads into the other
    __shared__ __align__(16) uint4 gAa[KG][BM * 8], gAb[KG][BM * 8], gWa[KG][BN * 4], gWb[KG][BN * 4], gHd[KG][BN];
    __shared__ __align__(16) uint2 gBs[KG][BM * 4];
    __shared__ __align__(16) float gDa[KG][BM];
    const int t = threadIdx.x & (NT - 1), lane = t & 63, c32 = lane & 31, h = lane >> 5;
    const int kg = KG == 1 ? 0 : __builtin_amdgcn_readfirstlane((int)threadIdx.x / NT);
    uint4 *const sAa = gAa[kg], *const sAb = gAb[kg], *const sWa = gWa[kg], *const sWb = gWb[kg], *const sHd = gHd[kg];
    uint2* const sBs = gBs[kg];
    float* const sDa = gDa[kg];
    const int wv = __builtin_amdgcn_readfirstlane(t >> 6), wm = wv / WN, wn = wv % WN;
    const int T = amv_xcd_tile(blockIdx.x, n_tw * n_z * n_tt);  // token tiles, weight tiles, k ranges
    const int tt = T % n_tt, tw = (T / n_tt) % n_tw, z = T / (n_tt * n_tw);
    const int n0 = tw * BN, m0 = tt * BM;
    const int K = nsb * 256;
    // the split's super-blocks, dealt to the KG groups of waves in runs of `run`; a group's turns past the end (or past the
    // split's) compute on the last super-block and add nothing
    const int z0 = z * sb_per, z_end = min(nsb, z0 + sb_per), run = (z_end - z0 + KG - 1) / KG;
    const int sb0 = z0 + run * kg, sb_end = min(z_end, sb0 + run), sb_last = z_end - 1;
    dst += (size_t)z * zstride;

    // rows past N and tokens past M read as zero
    const int mr = min(BM, M - m0), nr = min(BN, N - n0);
    const __amdgpu_buffer_rsrc_t ra = QG_RSRC(aq + (size_t)m0 * K, mr * K);
    const __amdgpu_buffer_rsrc_t rw = QG_RSRC(wq + (size_t)n0 * nsb * 8, nr * nsb * 128);
    const __amdgpu_buffer_rsrc_t rh = QG_RSRC(wh + (size_t)n0 * nsb, nr * nsb * 16);
    const __amdgpu_buffer_rsrc_t rs = QG_RSRC(as16 + (size_t)m0 * (K / 16), mr * (K / 4));
    const __amdgpu_buffer_rsrc_t rd = QG_RSRC(ad + (size_t)m0 * nsb, mr * nsb * 4);
    const uint32_t oa = (uint32_t)(t >> 3) * K + 16 * ((t & 7) ^ ((t >> 4) & 7));
    const uint32_t ow = (uint32_t)(t >> 2) * (nsb * 128) + 16 * ((t & 3) ^ ((t >> 4) & 3));
    const auto load = [&](uint4* sA, uint4* sW, int j, int half) {
#pragma unroll
        for (int i = 0; i < RA; ++i)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (qg_lds*)(sA + NT * i + 64 * wv), 16,
                                                     oa + (uint32_t)(NT / 8 * i) * K, 256 * j + 128 * half, 0, 0);
#pragma unroll
        for (int i = 0; i < RW; ++i)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rw, (qg_lds*)(sW + NT * i + 64 * wv), 16,
                                                     ow + (uint32_t)(NT / 4 * i) * (nsb * 128), 128 * j + 64 * half, 0, 0);
    };
    const auto load_head = [&](int j) {
        if (wv < BN / 64)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rh, (qg_lds*)(sHd + 64 * wv), 16, (uint32_t)t * (nsb * 16), 16 * j, 0,
                                                     0);
    };
    // activation sums (thread: token t / 4, 4 of the 16) and scale of super-block j, through registers
    typedef int v4i __attribute__((ext_vector_type(4)));
    v4i bs[RS];
    int da0;
    const auto load_sb = [&](int j) {
#pragma unroll
        for (int i = 0; i < RS; ++i)
            bs[i] = (v4i)__builtin_amdgcn_raw_buffer_load_b128(rs, (uint32_t)((t >> 2) + NT / 4 * i) * (K / 4) + 16 * (t & 3),
                                                               64 * j, 0);
        da0 = __builtin_amdgcn_raw_buffer_load_b32(rd, (uint32_t)min(t, BM - 1) * (nsb * 4), 4 * j, 0);
    };
    const auto store_sb = [&]() {
#pragma unroll
        for (int i = 0; i < RS; ++i)
            sBs[t + NT * i] = make_uint2(qg_h2(bs[i].x, bs[i].y), qg_h2(bs[i].z, bs[i].w));
        if (t < BM) sDa[t] = __int_as_float(da0);
    };

    qg_f16v acc[2];
    qg_v16i I1[2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][r] = 0.0f;

    const int ar = 64 * wm + c32, wr = 32 * wn + c32;
    const int ax = (c32 >> 1) & 7, wx = (c32 >> 2) & 3;  // the rows' XOR (64 wm, 32 i, 32 wn do not change them)
    const auto half_step = [&](const uint4* sA, const uint4* sW, uint32_t scw, bool first) {
#pragma unroll
        for (int cp = 0; cp < 2; ++cp) {
            const uint4 x = sW[wr * 4 + ((2 * cp + h) ^ wx)];
#pragma unroll
            for (int v = 0; v < 2; ++v) {
                const int u = 2 * cp + v;
                const qg_v4i B = v == 0 ? qg_v4i{(int)(x.x & 0x0F0F0F0Fu), (int)(x.y & 0x0F0F0F0Fu), (int)(x.z & 0x0F0F0F0Fu),
                                                 (int)(x.w & 0x0F0F0F0Fu)}
                                        : qg_v4i{(int)((x.x >> 4) & 0x0F0F0F0Fu), (int)((x.y >> 4) & 0x0F0F0F0Fu),
                                                 (int)((x.z >> 4) & 0x0F0F0F0Fu), (int)((x.w >> 4) & 0x0F0F0F0Fu)};
                const int sc = (int)((scw >> (8 * u)) & 0xFFu);
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    const uint4 a = sA[(ar + 32 * i) * 8 + ((2 * u + h) ^ ax)];
                    const qg_v16i zero = {};
                    const qg_v16i C = __builtin_amdgcn_mfma_i32_32x32x32_i8(
                        qg_v4i{(int)a.x, (int)a.y, (int)a.z, (int)a.w}, B, zero, 0, 0, 0);
                    if (first && u == 0) {
#pragma unroll
                        for (int r = 0; r < 16; ++r) I1[i][r] = __mul24(C[r], sc);
                    } else {
#pragma unroll
                        for (int r = 0; r < 16; ++r) I1[i][r] += __mul24(C[r], sc);
                    }
                }
                // one unit's results at a time (more do not fit the registers), added up here (the compiler would move
                // the additions behind the next barrier and keep the results until then)
                asm volatile("" : "+v"(I1[0]), "+v"(I1[1]));
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    };

    load_head(min(sb0, sb_last));
    load(sAa, sWa, min(sb0, sb_last), 0);
    load_sb(min(sb0, sb_last));
    QG_WAIT_LOADS();
    __syncthreads();
    for (int j = sb0; j < sb0 + run; ++j) {
        const int jn = min(j + 1, sb_last);
        load(sAb, sWb, min(j, sb_last), 1);
        const uint4 hd = sHd[wr];
        // scales and mins of units 0-3 and 4-7, one per byte
        const uint32_t sc0 = hd.y & 0x3F3F3F3Fu, sc1 = (hd.w & 0x0F0F0F0Fu) | ((hd.y >> 2) & 0x30303030u);
        const uint32_t mw = h ? ((hd.w >> 4) & 0x0F0F0F0Fu) | ((hd.z >> 2) & 0x30303030u) : hd.z & 0x3F3F3F3Fu;
        half_step(sAa, sWa, sc0, true);
        store_sb();
        QG_WAIT_LOADS();
        __syncthreads();
        load(sAa, sWa, jn, 0);
        load_head(jn);
        load_sb(jn);
        half_step(sAb, sWb, sc1, false);
        // end of super-block j: I2 (mins, each on its unit's two 16-sum slots, against the sums) and the f32 epilogue
        const qg_h8 Bmn = [&] {
            const uint32_t off = 0xE400E400u;  // -1024, -1024: 0x6400 | m is the f16 1024 + m
            typedef _Float16 h2 __attribute__((ext_vector_type(2)));
            qg_h8 r;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const uint32_t p = __builtin_amdgcn_perm(0x64646464u, mw, 0x04000400u + 0x00010001u * e);
                const h2 q = __builtin_bit_cast(h2, p) + __builtin_bit_cast(h2, off);
                r[2 * e] = q.x;
                r[2 * e + 1] = q.y;
            }
            return r;
        }();
        const float d = amv_h2f(hd.x), dm = amv_h2f(hd.x >> 16);
        if (KG == 1 || j < sb_end)
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int tl = 64 * wm + 32 * i;
            const qg_h8 Abs = *reinterpret_cast<const qg_h8*>(&sBs[(tl + c32) * 4 + 2 * h]);
            const qg_f16v zf = {};
            const qg_f16v I2 = __builtin_amdgcn_mfma_f32_32x32x16_f16(Abs, Bmn, zf, 0, 0, 0);
            if constexpr (SUMS) {
                const int n = n0 + wr;
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int m = m0 + tl + 4 * h + 8 * (r >> 2) + (r & 3);
                    if (m < M && n < N) {
                        int32_t* o = sums + (((size_t)m * N + n) * nsb + j) * 2;
                        o[0] = I1[i][r];
                        o[1] = (int)I2[r];
                    }
                }
            } else {
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const float4 v = *reinterpret_cast<const float4*>(&sDa[tl + 4 * h + 8 * q]);
                    const float da[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        acc[i][4 * q + r] = fmaf(fmaf(d, (float)I1[i][4 * q + r], -(dm * I2[4 * q + r])), da[r],
                                                 acc[i][4 * q + r]);
                }
            }
        }
        QG_WAIT_LOADS();
        __syncthreads();
    }
    qg_finish<SUMS, BM, NT, KG, ADD>(acc, gAa, kg, t, n0 + wr, m0 + 64 * wm + 4 * h, M, N, dst, ldd, add);
}

// ---------------------------------------------------------------------------------------------------------------
// Q6_K x Q8_K (reference vec_dot_q6_K_q8_K; ameva_qdecode.glsl:246-258 for the element layout). A super-block of 256
// is 16 sub-blocks of 16 consecutive elements with int8 scales sc_s and one f16 d: I = sum_s sc_s sum_k q_k a_k with
// q = (4 low bits from ql | 2 high bits from qh) - 32, dst += d_a d I. The sub-blocks are 16 long, so the matrix core
// runs v_mfma_i32_32x32x16_i8 (lane half h supplies 8 of the 16 bytes) and I accumulates sc_s C_s in integers. Step =
// one 128-element half n of the super-block: ql bytes 64 n .. + 63 and qh bytes 32 n .. + 31 give elements
// 128 n + {l, 32 + l, 64 + l, 96 + l} (l < 32) from ql[l] low / ql[32 + l] low / ql[l] high / ql[32 + l] high nibbles
// and qh[l] bits 0-1 / 2-3 / 4-5 / 6-7.
// ---------------------------------------------------------------------------------------------------------------
typedef long qg_i64;

#define QG6_LD (128 + 16)  // LDS row stride (bytes) of the 128-element steps

struct QgQ6Regs {
    uint4 l0, l1, qh;  // ql[16 hf ..], ql[32 + 16 hf ..], qh[16 hf ..] of the half (row t / 2, hf = t % 2)
    uint4 a0, a1, a2, a3;  // 64 activation int8 (token t / 2, elements 128 c + 64 hf ..)
    uint4 sc;          // at half 0: the row's 16 scales
    uint32_t d;        // at half 0: f16 d
    float da;          // at half 0: the token's d
};

template <int TT, int TW>
__device__ __forceinline__ void qg6_load(QgQ6Regs& s, int step, const uint4* __restrict__ wl,
                                         const uint4* __restrict__ wqh, const uint4* __restrict__ wsc,
                                         const uint16_t* __restrict__ wd, int N, int nsb, int n0,
                                         const int8_t* __restrict__ aq, const float* __restrict__ ad, int M, int m0,
                                         int K, int sb0) {
    constexpr int BN = 64 * TW, BM = 64 * TT;
    const int t = threadIdx.x, hf = t & 1;
    const int j = sb0 + (step >> 1), c = step & 1;
    if (t < 2 * BN) {
        const int row = min(n0 + (t >> 1), N - 1);
        const size_t sb = (size_t)row * nsb + j;
        s.l0 = wl[sb * 8 + 4 * c + hf];      // ql bytes 64 c + 16 hf
        s.l1 = wl[sb * 8 + 4 * c + 2 + hf];  // ql bytes 64 c + 32 + 16 hf
        s.qh = wqh[sb * 4 + 2 * c + hf];     // qh bytes 32 c + 16 hf
        if (c == 0) {
            s.sc = wsc[sb];
            s.d = wd[sb];
        }
    }
    if (t < 2 * BM) {
        const int tok = min(m0 + (t >> 1), M - 1);
        const uint4* p = reinterpret_cast<const uint4*>(aq + (size_t)tok * K + 256 * j + 128 * c + 64 * hf);
        s.a0 = p[0];
        s.a1 = p[1];
        s.a2 = p[2];
        s.a3 = p[3];
        if (c == 0) s.da = ad[(size_t)tok * nsb + j];
    }
}

// 4 bytes of ql nibbles n (already selected) and their 2 high bits hb (already at bit 4..5): n | hb - 32 per byte
__device__ __forceinline__ uint32_t qg6_q(uint32_t n, uint32_t hb) { return ((n | hb) + 0x60606060u) ^ 0x80808080u; }

template <int TT, int TW>
__device__ __forceinline__ void qg6_store(const QgQ6Regs& s, int step, int8_t* __restrict__ sW,
                                          int8_t* __restrict__ sA, int8_t* __restrict__ sSc, float* __restrict__ sD,
                                          float* __restrict__ sDa) {
    constexpr int BN = 64 * TW, BM = 64 * TT;
    const int t = threadIdx.x, hf = t & 1, c = step & 1;
    if (t < 2 * BN) {
        const int rl = t >> 1;
        uint4* d = reinterpret_cast<uint4*>(sW + rl * QG6_LD);
        const uint32_t L0[4] = {s.l0.x, s.l0.y, s.l0.z, s.l0.w}, L1[4] = {s.l1.x, s.l1.y, s.l1.z, s.l1.w};
        const uint32_t H[4] = {s.qh.x, s.qh.y, s.qh.z, s.qh.w};
        uint32_t q1[4], q2[4], q3[4], q4[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            q1[i] = qg6_q(L0[i] & 0x0F0F0F0Fu, (H[i] & 0x03030303u) << 4);
            q2[i] = qg6_q(L1[i] & 0x0F0F0F0Fu, (H[i] & 0x0C0C0C0Cu) << 2);
            q3[i] = qg6_q((L0[i] >> 4) & 0x0F0F0F0Fu, H[i] & 0x30303030u);
            q4[i] = qg6_q((L1[i] >> 4) & 0x0F0F0F0Fu, (H[i] >> 2) & 0x30303030u);
        }
        d[hf] = make_uint4(q1[0], q1[1], q1[2], q1[3]);      // elements 16 hf ..
        d[2 + hf] = make_uint4(q2[0], q2[1], q2[2], q2[3]);  // 32 + 16 hf ..
        d[4 + hf] = make_uint4(q3[0], q3[1], q3[2], q3[3]);  // 64 + 16 hf ..
        d[6 + hf] = make_uint4(q4[0], q4[1], q4[2], q4[3]);  // 96 + 16 hf ..
        if (c == 0) {  // scales of sub-blocks 8 hf .. 8 hf + 7 (bytes), d
            const uint32_t sw[2] = {hf ? s.sc.z : s.sc.x, hf ? s.sc.w : s.sc.y};
#pragma unroll
            for (int e = 0; e < 8; ++e) sSc[(8 * hf + e) * BN + rl] = (int8_t)((sw[e >> 2] >> (8 * (e & 3))) & 0xFFu);
            if (hf == 0) sD[rl] = amv_h2f(s.d);
        }
    }
    if (t < 2 * BM) {
        const int tl = t >> 1;
        uint4* d = reinterpret_cast<uint4*>(sA + tl * QG6_LD + 64 * hf);
        d[0] = s.a0;
        d[1] = s.a1;
        d[2] = s.a2;
        d[3] = s.a3;
        if (c == 0 && hf == 0) sDa[tl] = s.da;
    }
}

template <bool SUMS, int TT, int TW, bool ADD = false>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void k_qgemm_q6k(
    const uint4* __restrict__ wl, const uint4* __restrict__ wqh, const uint4* __restrict__ wsc,
    const uint16_t* __restrict__ wd, int N, int nsb, const int8_t* __restrict__ aq, const float* __restrict__ ad, int M,
    float* __restrict__ dst, int64_t ldd, const float* add, int32_t* __restrict__ sums, int sb_per, int64_t zstride, int n_tw, int n_tt,
    int n_z) {
    constexpr int BN = 64 * TW, BM = 64 * TT;
    __shared__ __align__(16) int8_t sW[2][BN * QG6_LD];
    __shared__ __align__(16) int8_t sA[2][BM * QG6_LD];
    __shared__ __align__(16) int8_t sSc[2][16 * BN];
    __shared__ __align__(16) float sD[2][BN], sDa[2][BM];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int wt = w & 1, ww = w >> 1, c32 = lane & 31, h = lane >> 5;
    const int T = amv_xcd_tile(blockIdx.x, n_tw * n_z * n_tt);  // token tiles, weight tiles, k ranges
    const int tt = T % n_tt, tw = (T / n_tt) % n_tw, z = T / (n_tt * n_tw);
    const int n0 = tw * BN, m0 = tt * BM;
    const int K = nsb * 256;
    const int sb0 = z * sb_per, sb_end = min(nsb, sb0 + sb_per);
    const int nsteps = (sb_end - sb0) * 2;
    dst += (size_t)z * zstride;

    qg_f16v acc[TT][TW];
    qg_v16i I[TT][TW];
#pragma unroll
    for (int i = 0; i < TT; ++i)
#pragma unroll
        for (int j = 0; j < TW; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                acc[i][j][r] = 0.0f;
                I[i][j][r] = 0;
            }

    QgQ6Regs st;
    qg6_load<TT, TW>(st, 0, wl, wqh, wsc, wd, N, nsb, n0, aq, ad, M, m0, K, sb0);
    qg6_store<TT, TW>(st, 0, sW[0], sA[0], sSc[0], sD[0], sDa[0]);
    __syncthreads();
    for (int step = 0; step < nsteps; ++step) {
        const int buf = step & 1, j = sb0 + (step >> 1), c = step & 1, jp = (step >> 1) & 1;
        if (step + 1 < nsteps) qg6_load<TT, TW>(st, step + 1, wl, wqh, wsc, wd, N, nsb, n0, aq, ad, M, m0, K, sb0);
#pragma unroll 2
        for (int u = 0; u < 8; ++u) {  // sub-block 8 c + u
            qg_i64 A[TT], B[TW];
            int sc[TW];
#pragma unroll
            for (int i = 0; i < TT; ++i)
                A[i] = *reinterpret_cast<const qg_i64*>(sA[buf] + (32 * (TT * wt + i) + c32) * QG6_LD + 16 * u + 8 * h);
#pragma unroll
            for (int jj = 0; jj < TW; ++jj) {
                const int rl = 32 * (TW * ww + jj) + c32;
                B[jj] = *reinterpret_cast<const qg_i64*>(sW[buf] + rl * QG6_LD + 16 * u + 8 * h);
                sc[jj] = sSc[jp][(8 * c + u) * BN + rl];
            }
#pragma unroll
            for (int i = 0; i < TT; ++i)
#pragma unroll
                for (int jj = 0; jj < TW; ++jj) {
                    const qg_v16i zero = {};
                    const qg_v16i C = __builtin_amdgcn_mfma_i32_32x32x16_i8(A[i], B[jj], zero, 0, 0, 0);
#pragma unroll
                    for (int r = 0; r < 16; ++r) I[i][jj][r] += __mul24(C[r], sc[jj]);
                }
        }
        if (c == 1) {  // end of super-block j
#pragma unroll
            for (int i = 0; i < TT; ++i) {
                const int tl = 32 * (TT * wt + i) + 4 * h;
                float da[16];
                if constexpr (!SUMS) {
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const float4 v = *reinterpret_cast<const float4*>(&sDa[jp][tl + 8 * q]);
                        da[4 * q] = v.x;
                        da[4 * q + 1] = v.y;
                        da[4 * q + 2] = v.z;
                        da[4 * q + 3] = v.w;
                    }
                }
#pragma unroll
                for (int jj = 0; jj < TW; ++jj) {
                    const int rl = 32 * (TW * ww + jj) + c32;
                    if constexpr (SUMS) {
                        const int n = n0 + rl;
#pragma unroll
                        for (int r = 0; r < 16; ++r) {
                            const int m = m0 + tl + 8 * (r >> 2) + (r & 3);
                            if (m < M && n < N) sums[((size_t)m * N + n) * nsb + j] = I[i][jj][r];
                        }
                    } else {
                        const float d = sD[jp][rl];
#pragma unroll
                        for (int r = 0; r < 16; ++r) acc[i][jj][r] = fmaf(d * da[r], (float)I[i][jj][r], acc[i][jj][r]);
                    }
#pragma unroll
                    for (int r = 0; r < 16; ++r) I[i][jj][r] = 0;
                }
            }
        }
        if (step + 1 < nsteps) {
            const int sp = ((step + 1) >> 1) & 1;
            qg6_store<TT, TW>(st, step + 1, sW[buf ^ 1], sA[buf ^ 1], sSc[sp], sD[sp], sDa[sp]);
            __syncthreads();
        }
    }
    if constexpr (!SUMS) {
#pragma unroll
        for (int jj = 0; jj < TW; ++jj) {
            const int n = n0 + 32 * (TW * ww + jj) + c32;
            if (n >= N) continue;
#pragma unroll
            for (int i = 0; i < TT; ++i)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int m = m0 + 32 * (TT * wt + i) + 8 * (r >> 2) + 4 * h + (r & 3);
                    if (m < M) {
                        const size_t o = (size_t)m * ldd + n;
                        if constexpr (ADD) dst[o] = acc[i][jj][r] + add[o];
                        else dst[o] = acc[i][jj][r];
                    }
                }
        }
    }
}

// ---------------------------------------------------------------------------------------------------------------
// host
// ---------------------------------------------------------------------------------------------------------------
// split of k shared with the f16 kernels (amv_mmq16.hip): workspace per device and the in-order partial sum
float* amv_splitk_workspace(size_t bytes, hipStream_t st);
int amv_splitk_count(int64_t tiles, int steps);
void amv_splitk_reduce(const float* part, int S, int64_t zstride, int64_t m, int64_t n, float* dst, int64_t ldd,
                       hipStream_t st, const float* add = nullptr);

// a launch's tiles and split of k (partials in the library's workspace, summed in order of k): k in units of `unit`
// blocks, `n_unit` of them
struct QgPlan {
    int n_tw, n_tt, S, per;
    float* out;
    int64_t ldo, zstride;
};
static int qg_plan(QgPlan& p, int bm, int bn, int64_t n_rows, int64_t m, int64_t k, int n_blk, int align, float* dst,
                   int64_t ldd, bool split, hipStream_t st) {
    p.n_tw = (int)((n_rows + bn - 1) / bn);
    p.n_tt = (int)((m + bm - 1) / bm);
    p.S = split ? amv_splitk_count((int64_t)p.n_tw * p.n_tt, (int)(k / 64)) : 1;
    p.per = n_blk;
    p.out = dst;
    p.ldo = ldd;
    p.zstride = 0;
    if (p.S > 1) {
        p.per = ((n_blk + p.S - 1) / p.S + align - 1) / align * align;
        p.S = (n_blk + p.per - 1) / p.per;
    }
    if (p.S > 1) {
        p.out = amv_splitk_workspace((size_t)p.S * m * n_rows * 4, st);
        if (!p.out) return AMV_ERR_HIP;  // never unsplit: the summation order would change
        p.ldo = n_rows;
        p.zstride = m * n_rows;
    }
    return AMV_OK;
}

struct QgCall {
    const void* w;
    int64_t n_rows, k;
    const void* act;
    int64_t m;
    float* dst;
    int64_t ldd;
    int32_t* sums;
    hipStream_t st;
    const float* add;
    bool split;  // k may be split over workgroups
};

// launches kernel<sums / plain / ADD> of a plan; A: the arguments after M
#define QG_GO(KERNEL, THREADS, ...)                                                                                       \
    do {                                                                                                                  \
        const dim3 grid((unsigned)((int64_t)p.n_tw * p.n_tt * p.S));                                                      \
        const float* kadd = p.S > 1 ? nullptr : c.add; /* with a split of k the residual joins in the partials' sum */    \
        const auto fn = c.sums ? KERNEL(true, false) : kadd ? KERNEL(false, true) : KERNEL(false, false);                 \
        hipLaunchKernelGGL(fn, grid, dim3(THREADS), 0, c.st, __VA_ARGS__, (int)c.m, p.out, p.ldo, kadd, c.sums, p.per,    \
                           p.zstride, p.n_tw, p.n_tt, p.S);                                                               \
        if (p.S > 1) amv_splitk_reduce(p.out, p.S, p.zstride, c.m, c.n_rows, c.dst, c.ldd, c.st, c.add);                  \
    } while (0)

template <int WT, int WM, int WN, int KG>
static int qg_block(const QgCall& c) {
    const int nb = (int)(c.k / 32);
    QgPlan p;
    const int rc = qg_plan(p, 64 * WM, 32 * WN, c.n_rows, c.m, c.k, nb, 4, c.dst, c.ldd, c.split, c.st);
    if (rc) return rc;
    const int8_t* aq = (const int8_t*)c.act;
    const int2* am = (const int2*)(aq + c.m * c.k);
    const uint8_t* wq = (const uint8_t*)c.w;
    const uint16_t* wd = (const uint16_t*)(wq + c.n_rows * nb * (WT == AMV_T_Q4_0 ? 16 : 32));
#define QG_K(SU, AD) k_qgemm<WT, SU, WM, WN, KG, AD>
    QG_GO(QG_K, 64 * WM * WN * KG, wq, wd, (int)c.n_rows, nb, aq, am);
#undef QG_K
    return AMV_OK;
}

template <int WM, int WN, int KG>
static int qg_q4k(const QgCall& c) {
    const int nsb = (int)(c.k / 256);
    QgPlan p;
    const int rc = qg_plan(p, 64 * WM, 32 * WN, c.n_rows, c.m, c.k, nsb, 1, c.dst, c.ldd, c.split, c.st);
    if (rc) return rc;
    const int8_t* aq = (const int8_t*)c.act;
    const uint4* wq = (const uint4*)c.w;
    const uint4* wh = (const uint4*)((const uint8_t*)c.w + c.n_rows * nsb * 128);
    const float* ad = (const float*)(aq + c.m * c.k);
    const int32_t* as16 = (const int32_t*)(aq + c.m * c.k + c.m * nsb * 4);
#define QG_K(SU, AD) k_qgemm_q4k<SU, WM, WN, KG, AD>
    QG_GO(QG_K, 64 * WM * WN * KG, wq, wh, (int)c.n_rows, nsb, aq, ad, as16);
#undef QG_K
    return AMV_OK;
}

// kg groups of waves (1, 2 or 4, at most MAX) share k
template <int WT, int WM, int WN, int MAX = 4>
static int qg_block_groups(const QgCall& c, int kg) {
    return kg == 1 ? qg_block<WT, WM, WN, 1>(c) : kg == 2 ? qg_block<WT, WM, WN, 2>(c) : qg_block<WT, WM, WN, MAX>(c);
}
template <int WM, int WN>
static int qg_q4k_groups(const QgCall& c, int kg) {
    return kg == 1 ? qg_q4k<WM, WN, 1>(c) : kg == 2 ? qg_q4k<WM, WN, 2>(c) : qg_q4k<WM, WN, 4>(c);
}

template <int TT, int TW>
static int qg_q6k(const QgCall& c) {  // ql [n][nsb][128] | qh [n][nsb][64] | scales [n][nsb][16] | d [n][nsb]
    const int nsb = (int)(c.k / 256);
    QgPlan p;
    const int rc = qg_plan(p, 64 * TT, 64 * TW, c.n_rows, c.m, c.k, nsb, 1, c.dst, c.ldd, c.split, c.st);
    if (rc) return rc;
    const int64_t nblk = c.n_rows * nsb;
    const uint8_t* base = (const uint8_t*)c.w;
    const uint4* wl = (const uint4*)base;
    const uint4* wqh = (const uint4*)(base + nblk * 128);
    const uint4* wsc = (const uint4*)(base + nblk * 192);
    const uint16_t* wd = (const uint16_t*)(base + nblk * 208);
    const int8_t* aq = (const int8_t*)c.act;
    const float* ad = (const float*)(aq + c.m * c.k);
#define QG_K(SU, AD) k_qgemm_q6k<SU, TT, TW, AD>
    QG_GO(QG_K, 256, wl, wqh, wsc, wd, (int)c.n_rows, nsb, aq, ad);
#undef QG_K
    return AMV_OK;
}
#undef QG_GO

// Whether k may be split over workgroups: not where 64 x 64 tiles alone give four workgroups per CU and the 128 x 128 ones
// are too few to be taken. Such a product fills the GPU with its wider tiles too (us, unsplit against 64 x 64 tiles staged
// through registers: 11000 x 6144 x 331 Q4_K 83 / 129, Q8_0 122 / 166, Q4_0 122 / 160; 16400 x 6144 x 200 83 / 125, 120 /
// 157, 116 / 155), and without the workspace it can overlap others on several streams and be a program's first product
// under capture.
static bool qg_may_split(int64_t n_rows, int64_t m) {
    return ((m + 127) / 128) * ((n_rows + 127) / 128) >= 384 || ((m + 63) / 64) * ((n_rows + 63) / 64) < 1024;
}

int amv_qgemm(int wtype, const void* w, int64_t n_rows, int64_t k, const void* act, int64_t m, float* dst, int64_t ldd,
              int32_t* sums, hipStream_t st, const float* add) {
    // Up to 64 tokens of Q4_0 / Q8_0 / Q4_K k stays whole: calls this small are made on several streams, which the split's
    // workspace does not allow at the same time.
    const QgCall c{w, n_rows, k, act, m, dst, ldd, sums, st, add,
                   !sums && (wtype == AMV_T_Q6_K || (m > 64 && qg_may_split(n_rows, m)))};
    const auto tiles = [&](int bm, int bn) { return ((m + bm - 1) / bm) * ((n_rows + bn - 1) / bn); };
    const auto wgs = [&](int bm, int bn) {  // workgroups with the split of k
        return tiles(bm, bn) * (c.split ? amv_splitk_count(tiles(bm, bn), (int)(k / 64)) : 1);
    };
    // 64 x 64 tiles with four groups sharing k while that leaves at most one workgroup per CU, then 64 x 128 with four (two
    // where LDS holds no more, or from one to two workgroups per CU), then a group to a workgroup on 128 x 128 (Q4_K below 384
    // of them: 64 x 128; Q4_0 below that and without a split of k: 64 x 128, two groups). Measured (us; before: tiles staged through registers, 4 waves each,
    // m <= 64 on 16 x 16 tiles):
    //   rows x k, tokens     Q4_K           Q8_0           Q4_0
    //   14336 x 4096,  48    18 (48)        22 (111)       22 (116)
    //   4096 x 14336,  48    48 (173)       61 (373)       63 (395)     (split over workgroups 22, 24, 24)
    //   4096 x 4096,   96    16 (38)        19 (39)        21 (42)
    //   14336 x 4096, 128    27 (46)        35 (51)        33 (52)
    //   4096 x 4096,  512    29 (47)        39 (56)        39 (56)
    //   14336 x 4096, 331    61 (94)        82 (122)       79 (114)
    //   4096 x 14336, 331    67 (96)        76 (120)       81 (111)
    //   14336 x 4096, 512    78 (97)        93 (117)       98 (110)
    //   28672 x 4096, 512    158 (199)      187 (228)      195 (225)
    // The neighbours of a choice: 14336 x 128 rows of Q4_K 35 with 64 x 64 tiles (448 of them), 6144 x 128 24 with 64 x 128
    // (17 with 64 x 64), 4096 x 512 41 with one group (29 with four).
    const bool t64 = wgs(64, 64) <= 256, t128 = wgs(64, 128) <= 256, two = wgs(64, 128) <= 512, big = tiles(128, 128) >= 384;
    // No more groups than k has steps (Q4_K: super-blocks) for: those without cost their turns and the joining of the sums
    // (us, 4096 x 256 with 65 / 512 tokens, four groups in brackets: Q4_K 6.0 (8.2) / 7.7 (12.7), Q4_0 6.1 (6.9) / 8.2 (10.4);
    // 4096 x 768 of Q4_K keeps four: 8.2, two 8.9).
    const int64_t units = wtype == AMV_T_Q4_K ? k / 256 : (k + 127) / 128;
    const int kg = units >= 3 ? 4 : (int)units, kg2 = std::min(kg, 2);
    int rc;
    if (wtype == AMV_T_Q4_K)
        rc = t64    ? qg_q4k_groups<1, 2>(c, kg)
             : t128 ? qg_q4k_groups<1, 4>(c, kg)
             : two  ? qg_q4k_groups<1, 4>(c, kg2)
             : big  ? qg_q4k<2, 4, 1>(c)
                    : qg_q4k<1, 4, 1>(c);
    else if (wtype == AMV_T_Q4_0)
        rc = t64                               ? qg_block_groups<AMV_T_Q4_0, 1, 2>(c, kg)
             : t128                            ? qg_block_groups<AMV_T_Q4_0, 1, 4>(c, kg)
             : big || (c.split && k >= 6144)   ? qg_block<AMV_T_Q4_0, 2, 4, 1>(c)
                                               : qg_block_groups<AMV_T_Q4_0, 1, 4>(c, kg2);
    else if (wtype == AMV_T_Q8_0)
        rc = t64 ? qg_block_groups<AMV_T_Q8_0, 1, 2>(c, kg)
             : t128 ? qg_block_groups<AMV_T_Q8_0, 1, 4, 2>(c, kg2)
                    : qg_block<AMV_T_Q8_0, 2, 4, 1>(c);
    else
        rc = big ? qg_q6k<2, 2>(c) : qg_q6k<1, 1>(c);
    if (rc) return rc;
    return amv_check_launch("amv_mul_mat_q_act");
}
