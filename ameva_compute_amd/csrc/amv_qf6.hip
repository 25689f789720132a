// Prefill MUL_MAT of Q4_0 weights on the scaled 6-bit matrix instruction of MI355X, ggml's block integers exact.
//
// Same product as k_qgemm (amv_qgemm.hip): dst[m][n] = sum_b S_b (d_w d_a), S_b = sum_k (nib_k - 8) q_k, with the same
// f32 operation per block: where the blocks are summed in the same order the two kernels' results are equal bit for
// bit. What bounds k_qgemm is the f32 epilogue of each 32-block beside the matrix core (convert, scale product, fma: 48
// VALU operations per 32 x 32 tile and block). Here two of the three are gone:
//   * S_b comes out of v_mfma_scale_f32_32x32x64_f8f6f4 as f32. A 6-bit E2M3 code c < 16 is the number c / 8, so a
//     nibble is its own code; the int8 activation is two digits, q = 16 (q >> 4) + (q & 15), both within the codes
//     -8 .. 15. The 64 k slots of one instruction are the block's 32 elements twice: lane half 0 multiplies the weights
//     with the high digits, half 1 with the low ones, the power of two of each digit in the block exponents. The sums
//     stay below 2^24: exact. The offset -8 sum(q) enters as the C operand (one value per token, so one per lane).
//   * d_w d_a is the outer product of two vectors: one v_mfma_f32_32x32x1_2b_f32 gives it for two tiles, each value
//     one f32 product, as the VALU would.
// With registers only (2 waves per SIMD) a tile and block take 75 cycles in this form and 150 in the int8 one; the
// kernel runs at ~215 (28 VALU operations and 64 matrix-core cycles per tile and block, the rest LDS latency, barriers
// and the last round of tiles), k_qgemm at ~260.
//
// The digits are made once per activation (k_f6_pack, ~3 us) into the scratch part of AMV_ACT_Q8_0_F6; weights are
// unpacked at staging: 16 nibbles (two dwords) spread to 16 6-bit fields (three dwords) in 10 operations, in an order
// that the digits follow (f6_elem).
//
// Tiling: 4 waves on 128 tokens x 128 weight rows; a wave owns 32 tokens x 4 tiles of 32 rows, so the C operand (16 moves)
// serves 4 tiles. A = weight rows, B = tokens: lane l of the result holds token l % 32 and rows 8 (r / 4) + 4 (l / 32)
// + r % 4. Steps of 64 k, double-buffered in LDS. A workgroup alone on its CU spends its time waiting for loads (1.1 us a
// step of 2600 cycles with both operands one step ahead in registers, 0.7 with the scheme below), so the weights run
// four steps ahead in registers and the digits, which need no unpacking, go to LDS directly. Grid order and the split
// of k as k_qgemm.
#include "amv_common.h"

#include <algorithm>

typedef int f6_v8i __attribute__((ext_vector_type(8)));
typedef unsigned int f6_v4u __attribute__((ext_vector_type(4)));
typedef float f6_v16 __attribute__((ext_vector_type(16)));
typedef float f6_v32 __attribute__((ext_vector_type(32)));

#define BM 128  // tokens and weight rows of a tile
#define BN 128
#define TW 4    // 32-row tiles of a wave
#define F6_FMT 2  // E2M3
// block exponents: a code unit is 2^-3, the high digit counts 16
#define F6_EXP_LO (127 + 3)
#define F6_EXP_HI (127 + 3 + 4)

// 16 nibbles (a's, then b's) to 16 6-bit fields: field f holds nibble f6_nib(f) of the 16. Nibble j of a dword sits at
// bit 4 j; fields whose bit 6 f falls on a nibble's own bit or two above it take that nibble, so two masks per output
// dword do; a's last nibble crosses into the second dword.
__device__ __forceinline__ void f6_spread(uint32_t a, uint32_t b, int& d0, int& d1, int& d2) {
    const uint32_t a2 = a << 2, b2 = b << 2;
    d0 = (int)((a & 0x0F00F00Fu) | (a2 & 0xC03C03C0u));
    d1 = (int)((b & 0xF00F00F0u) | (b2 & 0x03C03C00u) | (a >> 30));
    d2 = (int)((a & 0x00F00F00u) | (b2 & 0x3C03C03Cu));
}
// the element (0..31 of the block) in field f of a row's 32 fields: dword d of the block's 16 bytes holds elements
// 4 d + j / 2 (j even) and 16 + 4 d + j / 2 (j odd); fields 0..15 come from dwords 0, 1, fields 16..31 from 2, 3
__host__ __device__ constexpr int f6_elem(int f) {
    constexpr int nib[16] = {0, 1, 3, 4, 6, 7, 8 + 1, 8 + 2, 8 + 4, 8 + 5, 8 + 7, 8 + 0, 2, 8 + 3, 5, 8 + 6};
    const int s = nib[f & 15], d = 2 * (f >> 4) + (s >> 3), j = s & 7;
    return 4 * d + (j >> 1) + ((j & 1) ? 16 : 0);
}

// one thread per (token, block): the block's 32 int8 as high and low digits (192 bits each, fields in f6_elem's order),
// stored as 16 + 8 bytes in the layouts the MFMA operand reads want: hi4/lo4 [block][token][2] uint4, [..][2] uint2,
// and {d, -8 sum} [block][token]. Tokens m .. mp - 1 are zero. 4 consecutive threads take 4 blocks of one token (128
// contiguous bytes).
__global__ __launch_bounds__(256) void k_f6_pack(const int8_t* __restrict__ aq, const int2* __restrict__ am, int m,
                                                int mp, int nb, uint4* __restrict__ d16, uint2* __restrict__ d8,
                                                float2* __restrict__ meta) {
    const int tok = (int)blockIdx.x * 64 + (threadIdx.x >> 2), b = (int)blockIdx.y * 4 + (threadIdx.x & 3);
    if (b >= nb || tok >= mp) return;
    uint32_t hi[6] = {}, lo[6] = {};
    float2 mt = make_float2(0.0f, 0.0f);
    if (tok < m) {
        const uint4* p = reinterpret_cast<const uint4*>(aq + (size_t)tok * nb * 32 + 32 * (size_t)b);
        const uint4 x = p[0], y = p[1];
        const int2 s = am[(size_t)tok * nb + b];
        mt = make_float2(__int_as_float(s.x), (float)(-8 * s.y));
        const uint32_t v[8] = {x.x, x.y, x.z, x.w, y.x, y.y, y.z, y.w};
#pragma unroll
        for (int f = 0; f < 32; ++f) {
            const int e = f6_elem(f);
            const int q = (int)(v[e >> 2] << (24 - 8 * (e & 3))) >> 24, h = q >> 4;
            const uint32_t hc = h < 0 ? (uint32_t)(32 - h) : (uint32_t)h, lc = (uint32_t)(q & 15);  // sign, magnitude
            const int w = (6 * f) >> 5, sh = (6 * f) & 31;
            hi[w] |= hc << sh;
            lo[w] |= lc << sh;
            if (sh > 26) {
                hi[w + 1] |= hc >> (32 - sh);
                lo[w + 1] |= lc >> (32 - sh);
            }
        }
    }
    const size_t o = ((size_t)b * mp + tok) * 2;
    d16[o] = make_uint4(hi[0], hi[1], hi[2], hi[3]);
    d16[o + 1] = make_uint4(lo[0], lo[1], lo[2], lo[3]);
    d8[o] = make_uint2(hi[4], hi[5]);
    d8[o + 1] = make_uint2(lo[4], lo[5]);
    meta[o >> 1] = mt;
}

// one thread's weight block of a step (row, block): the 16 nibble bytes and the scale's f16 bits
struct F6W {
    f6_v4u w;
    uint32_t dw;
};

typedef __attribute__((address_space(3))) void f6_lds;
// wait until at most n vector memory loads are outstanding (n < 16; the other counters are left alone)
#define F6_WAIT(n) __builtin_amdgcn_s_waitcnt(0x0f70 | (n))

template <bool SUMS, bool ADD>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void k_qgemm_f6(
    const uint8_t* __restrict__ wq, const uint16_t* __restrict__ wd, int N, int nb, const uint4* __restrict__ d16,
    const uint2* __restrict__ d8, const float2* __restrict__ meta, int mp, int M, float* __restrict__ dst, int64_t ldd,
    const float* add, int32_t* __restrict__ sums, int vec, int kb_per, int64_t zstride, int n_tw, int n_tt, int n_z) {
    // the two buffers of a step are variables of their own, so that the compiler sees that reads of one do not wait for
    // the loads into the other
    __shared__ __align__(16) uint4 sA16a[4 * BM], sA16b[4 * BM], sW16a[2 * BN], sW16b[2 * BN];
    __shared__ __align__(16) uint2 sA8a[4 * BM], sA8b[4 * BM], sW8a[2 * BN], sW8b[2 * BN];
    __shared__ __align__(16) float2 sMta[2 * BM], sMtb[2 * BM];
    __shared__ __align__(16) float sDwa[2 * BN], sDwb[2 * BN];
    const int t = threadIdx.x, lane = t & 63, wv = __builtin_amdgcn_readfirstlane(t >> 6), c = lane & 31, h = lane >> 5;
    const int wm = wv;
    // tile index: token tile fastest, then the split of k, then the weight tile
    const int T = amv_xcd_tile(blockIdx.x, n_tw * n_z * n_tt);
    const int tt = T % n_tt, tw = (T / n_tt) % n_tw, z = T / (n_tt * n_tw);
    const int n0 = tw * BN, m0 = tt * BM;
    const int b0 = z * kb_per, b_end = min(nb, b0 + kb_per);
    const int nsteps = (b_end - b0 + 1) / 2;
    dst += (size_t)z * zstride;

    f6_v16 acc[TW];
#pragma unroll
    for (int j = 0; j < TW; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[j][r] = 0.0f;

    // Weights run four steps ahead in registers (a row's 32 bytes of a step are a quarter of a line, so this is the line
    // being fetched once, early); digits go to LDS without registers, one step ahead. Buffer loads: the per-thread
    // offsets are fixed, the step is a scalar, and rows past N read as zero. A buffer's range check leaves out the scalar
    // offset: each step's weights have a buffer that begins at its first block (an odd last step reads the next row's
    // first block as its second, zero behind the last row), and the digits' block index stays below b_end. That second
    // block is not computed.
    F6W sw0, sw1, sw2, sw3;
    const int blk = t & 1, wrow = t >> 1;
    const uint8_t* const pw = wq + ((size_t)n0 * nb + b0) * 16;
    const uint32_t wbytes = ((uint32_t)min(BN, N - n0) * nb - b0) * 16u;
    const __amdgpu_buffer_rsrc_t rd =
        __builtin_amdgcn_make_buffer_rsrc((void*)wd, 0, (uint32_t)N * (uint32_t)nb * 2u, 0x00027000);
    const uint32_t ow = ((uint32_t)wrow * nb + blk) * 16u;
    const int srow = min(n0 + wrow, N - 1);  // scales of a row pair side by side, an odd last row by itself
    const uint32_t od = (uint32_t)amv_q4_0_didx(srow, b0 + blk, nb, N) * 2u, sd = srow < (N & ~1) ? 8u : 4u;
    const auto load_w = [&](F6W& g, int step) {
        const int s = min(step, nsteps - 1);
        const __amdgpu_buffer_rsrc_t rw =
            __builtin_amdgcn_make_buffer_rsrc((void*)(pw + s * 32), 0, wbytes - s * 32, 0x00027000);
        g.w = __builtin_amdgcn_raw_buffer_load_b128(rw, ow, 0, 0);
        g.dw = __builtin_amdgcn_raw_buffer_load_b16(rd, od + (uint32_t)s * sd, 0, 0);
        __builtin_amdgcn_sched_barrier(0);  // not after the step's arithmetic, where the compiler would put them
    };
    // the step's digits, copied as they lie (BM tokens of two blocks), each wave a quarter
    const uint64_t region = (uint64_t)mp * nb;
    const __amdgpu_buffer_rsrc_t r16 =
        __builtin_amdgcn_make_buffer_rsrc((void*)d16, 0, (uint32_t)(region * 32), 0x00027000);
    const __amdgpu_buffer_rsrc_t r8 = __builtin_amdgcn_make_buffer_rsrc((void*)d8, 0, (uint32_t)(region * 16), 0x00027000);
    const __amdgpu_buffer_rsrc_t rm = __builtin_amdgcn_make_buffer_rsrc((void*)meta, 0, (uint32_t)(region * 8), 0x00027000);
    const auto load_d = [&](uint4* a16, uint2* a8, float2* mt, int step) {
        const int s = min(step, nsteps - 1), b = b0 + 2 * s, b1 = min(b + 1, b_end - 1);
        const uint32_t at[2] = {(uint32_t)b * (uint32_t)mp + (uint32_t)m0,  // (block, token) index
                                (uint32_t)b1 * (uint32_t)mp + (uint32_t)m0};
#pragma unroll
        for (int bl = 0; bl < 2; ++bl) {
            const uint32_t ab = at[bl];
            // BM * 32 bytes of a block, 1 KB per wave; BM * 8, 256 per wave
            __builtin_amdgcn_raw_ptr_buffer_load_lds(r16, (f6_lds*)(a16 + bl * 2 * BM + 64 * wv), 16, 16 * t, ab * 32u, 0, 0);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rm, (f6_lds*)(mt + bl * BM + 32 * wv), 4, 4 * t, ab * 8u, 0, 0);
        }
        // BM * 16 bytes per block: the two blocks' 1 KB pieces dealt to the waves
        __builtin_amdgcn_raw_ptr_buffer_load_lds(r8, (f6_lds*)(a8 + 128 * wv), 16, 16 * lane + 1024 * (wv & 1),
                                                 (wv >> 1 ? at[1] : at[0]) * 16u, 0, 0);
        __builtin_amdgcn_sched_barrier(0);  // these before the step's weight loads: the wait below counts on it
    };
    const auto store = [&](const F6W& g, uint4* w16, uint2* w8, float* dw) {
        int d[6];
        f6_spread(g.w.x, g.w.y, d[0], d[1], d[2]);
        f6_spread(g.w.z, g.w.w, d[3], d[4], d[5]);
        w16[blk * BN + wrow] = make_uint4(d[0], d[1], d[2], d[3]);
        w8[blk * BN + wrow] = make_uint2(d[4], d[5]);
        dw[blk * BN + wrow] = amv_h2f((uint16_t)g.dw);
    };
    const int ea = F6_EXP_LO, eb = h ? F6_EXP_LO : F6_EXP_HI;  // half 0: the high digits
    const auto compute = [&](int step, const uint4* a16, const uint2* a8, const float2* mt,
                             const uint4* w16, const uint2* w8, const float* dw) {
        const bool one = b0 + 2 * step + 1 == b_end;
#pragma unroll 1
        for (int bl = 0; bl < 2; ++bl) {
            if (bl && one) break;  // (a variable count of blocks compiles to a slower loop)
            const int tok = 32 * wm + c;
            const uint4 b4 = a16[(bl * BM + tok) * 2 + h];
            const uint2 b2 = a8[(bl * BM + tok) * 2 + h];
            const float2 ms = mt[bl * BM + tok];
            const f6_v8i B = {(int)b4.x, (int)b4.y, (int)b4.z, (int)b4.w, (int)b2.x, (int)b2.y, 0, 0};
            f6_v16 C0;
#pragma unroll
            for (int r = 0; r < 16; ++r) C0[r] = ms.y;
#pragma unroll
            for (int p = 0; p < TW / 2; ++p) {
                f6_v32 o;
                if constexpr (!SUMS) {
                    const f6_v32 zero = {};
                    o = __builtin_amdgcn_mfma_f32_32x32x1f32(dw[bl * BN + 64 * p + lane], ms.x, zero, 0, 0, 0);
                }
#pragma unroll
                for (int jj = 0; jj < 2; ++jj) {
                    const int j = 2 * p + jj, rl = 32 * j + c;
                    const uint4 a4 = w16[bl * BN + rl];
                    const uint2 a2 = w8[bl * BN + rl];
                    const f6_v8i A = {(int)a4.x, (int)a4.y, (int)a4.z, (int)a4.w, (int)a2.x, (int)a2.y, 0, 0};
                    const f6_v16 P = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(A, B, C0, F6_FMT, F6_FMT, 0, ea, 0,
                                                                                     eb);
                    if constexpr (SUMS) {
                        const int b = b0 + 2 * step + bl, m = m0 + tok;
#pragma unroll
                        for (int r = 0; r < 16; ++r) {
                            const int n = n0 + 32 * j + 8 * (r >> 2) + 4 * h + (r & 3);
                            if (m < M && n < N) sums[((size_t)m * N + n) * nb + b] = (int32_t)P[r];
                        }
                    } else {
#pragma unroll
                        for (int r = 0; r < 16; ++r) acc[j][r] = fmaf(P[r], o[16 * jj + r], acc[j][r]);
                    }
                }
            }
        }
    };
    load_d(sA16a, sA8a, sMta, 0);
    load_w(sw0, 0);
    load_w(sw1, 1);
    load_w(sw2, 2);
    load_w(sw3, 3);
    store(sw0, sW16a, sW8a, sDwa);
    F6_WAIT(6);  // the digits; the three later weight blocks (two loads each) may be out
    __syncthreads();
    // step u of four: digits of step + 1 to the other buffer, weights of step + 4 to the registers just free; then
    // step + 1's weights to LDS. At the wait the two weight loads of this step may be out, the digits before them not.
#define F6_STEP(u, W, WN1, X, Y)                                                       \
    load_d(sA16##Y, sA8##Y, sMt##Y, s0 + u + 1);                           \
    load_w(W, s0 + u + 4);                                                             \
    compute(s0 + u, sA16##X, sA8##X, sMt##X, sW16##X, sW8##X, sDw##X); \
    if (s0 + u + 1 >= nsteps) break;                                                   \
    store(WN1, sW16##Y, sW8##Y, sDw##Y);                                               \
    F6_WAIT(2);                                                                        \
    __syncthreads();
    for (int s0 = 0;; s0 += 4) {
        F6_STEP(0, sw0, sw1, a, b)
        F6_STEP(1, sw1, sw2, b, a)
        F6_STEP(2, sw2, sw3, a, b)
        F6_STEP(3, sw3, sw0, b, a)
    }
#undef F6_STEP
    F6_WAIT(0);  // the last step's prefetch may still write LDS
    if constexpr (!SUMS) {
        const int m = m0 + 32 * wm + c;
        if (m >= M) return;
        float* drow = dst + (size_t)m * ldd;
        const float* arow = ADD ? add + (size_t)m * ldd : nullptr;
#pragma unroll
        for (int j = 0; j < TW; ++j)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int n = n0 + 32 * j + 8 * q + 4 * h;
                float4 v = make_float4(acc[j][4 * q], acc[j][4 * q + 1], acc[j][4 * q + 2], acc[j][4 * q + 3]);
                if (vec && n + 3 < N) {
                    if constexpr (ADD) {
                        const float4 e = *reinterpret_cast<const float4*>(arow + n);
                        v = make_float4(v.x + e.x, v.y + e.y, v.z + e.z, v.w + e.w);
                    }
                    *reinterpret_cast<float4*>(drow + n) = v;
                } else {
                    const float u[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        if (n + r < N) drow[n + r] = ADD ? u[r] + arow[n + r] : u[r];
                }
            }
    }
}

// ---------------------------------------------------------------------------------------------------------------
// host
// ---------------------------------------------------------------------------------------------------------------
float* amv_splitk_workspace(size_t bytes, hipStream_t st);
int amv_splitk_count(int64_t tiles, int steps);
bool amv_qgemm_may_split(int64_t n_rows, int64_t m);
void amv_splitk_reduce(const float* part, int S, int64_t zstride, int64_t m, int64_t n, float* dst, int64_t ldd,
                       hipStream_t st, const float* add = nullptr);

static int f6_launch(const void* w, int64_t n_rows, int64_t k, uint8_t* act, int64_t m, float* dst, int64_t ldd,
                     int32_t* sums, hipStream_t st, const float* add) {
    const int nb = (int)(k / 32);
    const int n_tw = (int)((n_rows + BN - 1) / BN), n_tt = (int)((m + BM - 1) / BM);
    const int64_t tiles = (int64_t)n_tw * n_tt;
    int S = sums || !amv_qgemm_may_split(n_rows, m) ? 1 : amv_splitk_count(tiles, (nb + 1) / 2), per = nb;
    float* out = dst;
    int64_t ldo = ldd, zstride = 0;
    if (S > 1) {
        per = ((nb + S - 1) / S + 1) & ~1;
        S = (nb + per - 1) / per;
        if (S > 1) {
            out = amv_splitk_workspace((size_t)S * m * n_rows * 4, st);
            if (!out) return AMV_ERR_HIP;  // never unsplit: the summation order would change
            ldo = n_rows;
            zstride = m * n_rows;
        } else {
            per = nb;
        }
    }
    const AmvQ80F6 L = amv_q8_0_f6_layout(m, k);
    const uint4* d16 = (const uint4*)(act + L.d16);
    const uint2* d8 = (const uint2*)(act + L.d8);
    const float2* meta = (const float2*)(act + L.meta);
    const uint8_t* wq = (const uint8_t*)w;
    const uint16_t* wd = (const uint16_t*)(wq + n_rows * nb * 16);
    const float* kadd = S > 1 ? nullptr : add;  // with a split of k the residual joins in the sum of the partials
    const int vec = ldo % 4 == 0 && ((uintptr_t)out & 15) == 0 && ((uintptr_t)kadd & 15) == 0;
    const dim3 grid((unsigned)(tiles * S));
#define F6_GO(SU, AD)                                                                                              \
    hipLaunchKernelGGL((k_qgemm_f6<SU, AD>), grid, dim3(256), 0, st, wq, wd, (int)n_rows, nb, d16, d8, meta, \
                       (int)L.mp, (int)m, out, ldo, kadd, sums, vec, per, zstride, n_tw, n_tt, S)
    if (sums) F6_GO(true, false);
    else if (kadd) F6_GO(false, true);
    else F6_GO(false, false);
#undef F6_GO
    if (S > 1) amv_splitk_reduce(out, S, zstride, m, n_rows, dst, ldd, st, add);
    return AMV_OK;
}

int amv_qgemm(int wtype, const void* w, int64_t n_rows, int64_t k, const void* act, int64_t m, float* dst, int64_t ldd,
              int32_t* sums, hipStream_t st, const float* add);

// Q4_0 weights with an AMV_ACT_Q8_0_F6 activation of m rows: its plain Q8_0 prefix is packed into its scratch part, then
// the product
int amv_qgemm_f6(const void* w, int64_t n_rows, int64_t k, void* act, int64_t m, float* dst, int64_t ldd, int32_t* sums,
                 hipStream_t st, const float* add) {
    const int nb = (int)(k / 32);
    const int64_t tiles = ((m + BM - 1) / BM) * ((n_rows + BN - 1) / BN);
    // fewer than 1.5 workgroups per CU: the int8 kernel, whose smaller tiles share k between groups of waves (6144 x 4096 x
    // 512 57 us against 73, 4096 x 4096 x 96 21 against 69). Measured here against it (us): 28672 x 4096 x 512 184 (195),
    // 14336 x 4096 x 512 97 (98), 4096 x 14336 x 512 106 (114).
    if (tiles * (sums || !amv_qgemm_may_split(n_rows, m) ? 1 : amv_splitk_count(tiles, (nb + 1) / 2)) < 384)
        return amv_qgemm(AMV_T_Q4_0, w, n_rows, k, act, m, dst, ldd, sums, st, add);
    uint8_t* a = (uint8_t*)act;
    const AmvQ80F6 L = amv_q8_0_f6_layout(m, k);
    hipLaunchKernelGGL(k_f6_pack, dim3((unsigned)((L.mp + 63) / 64), (unsigned)((nb + 3) / 4)), dim3(256), 0, st,
                       (const int8_t*)a, (const int2*)(a + m * k), (int)m, (int)L.mp, nb, (uint4*)(a + L.d16),
                       (uint2*)(a + L.d8), (float2*)(a + L.meta));
    const int rc = f6_launch(w, n_rows, k, a, m, dst, ldd, sums, st, add);
    if (rc) return rc;
    return amv_check_launch("amv_mul_mat_q_act");
}
