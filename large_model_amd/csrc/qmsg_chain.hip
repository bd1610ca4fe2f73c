/* qmsg_chain.hip - rows as one fp32 FMA chain in element order, on the fp32 matrix cores.
 *
 * The reference's matmul_exact (src/quant.c:97-115) dots a row dequantised to fp32
 * (qms_dequant_row, src/quant.c:17-93) with an fp32 input row: acc = fma(w_i, x_i, acc), i
 * ascending. Its --exact mode takes every product that way, and every mode the F16 and Q8_0
 * matrices (outside qms_fast_supported) and the calls that hold one.
 *
 * v_mfma_f32_16x16x4_f32 is that chain: each of its 16 x 16 results is fma(a_3, b_3, fma(a_2,
 * b_2, fma(a_1, b_1, fma(a_0, b_0, c)))), rounded after every step, with subnormals, infinities
 * and NaN as the scalar fma has them (compared bit for bit with host fmaf on the device over
 * normals, wide exponents, subnormals and non-finite values). So one instruction of 32 cycles
 * advances 16 rows x 16 input rows by four elements, twice the rate of the vector ALU, which is
 * free to dequantise meanwhile.
 *
 * A wave takes 16 rows x 16 NC input rows, a block four waves that share the inputs in LDS.
 * Each wave streams its own rows: chunks of contiguous row bytes in 16-byte loads (a lane per
 * (row, quarter of a 32-block) straight from memory made so many small requests that the 30B
 * Q8_0 gate/up stayed at 1 TB/s), through a wave-private LDS buffer, so the weights need no block
 * barrier. The instruction wants element 4j + g of a 32-block (j = 0..7) in lane group g =
 * lane / 16; lane (row, g) reads a quarter of the block and the four lanes of a row trade bytes
 * with the lane-swap instructions. Inputs sit in LDS as [row][block][g][8]: all of them before
 * the loop where they fit (RES), else a few blocks at a time with one barrier each.
 *
 * Bound: at one token the one chain's latency. At batch sizes no unit is full (30B, Q8_0, 201 tokens
 * of a skewed load, gate/up / down): the matrix pipe is busy 0.49 / 0.44 of the time, partly filled
 * 16-column tiles included, LDS 0.37 / 0.35, over half of that bank conflicts (inputs are stored as
 * single words); two blocks per CU leave 1.7 waves per SIMD, which wait to issue for 0.64 / 0.60 of
 * their cycles. The 30B shape with Q8_0 experts, us, against one lane per row
 * and four slots per pass on the vector ALU: gate/up with SwiGLU 19 (45 + 7), down 9.8 (20) at
 * one token; 254 and 135 (together 5744) at 201 tokens of a skewed load, the layer 383 (5860). */
#include <type_traits>

#include "qmsg_device.h"

namespace qmsg {

namespace {

constexpr int kChRows = 64;               /* rows of a block                                    */
constexpr int kChResFloats = 16 * 1024;   /* inputs of up to 64 KiB are staged whole            */
constexpr size_t kChResLds = 80 * 1024;   /* expert rows: where two blocks still share a CU     */

/* A wave's staged chunk: NB blocks of 16 rows, BYTES per row, moved as 16-byte units to LDS rows
 * RS bytes apart (RS / 4 mod 64 a multiple of 4 that 16 rows spread over the banks). */
template <int TYPE>
struct ChFmt {
    static constexpr int NB = TYPE == 0 ? 2 : (TYPE == 1 ? 4 : 8);
    static constexpr int BYTES = TYPE == 0 || TYPE == 1 ? 256 : (TYPE == 8 ? 272 : (TYPE == 14 ? 210 : (TYPE == 3 ? 160 : 144)));
    static constexpr int UNITS = (BYTES + 15) / 16;
    static constexpr int RS = TYPE == 0 || TYPE == 1 || TYPE == 8 ? 272 : (TYPE == 14 ? 240 : (TYPE == 3 ? 176 : 144));
    static constexpr int NL = (16 * UNITS + 63) / 64;           /* loads per lane and chunk       */
    static constexpr int XB = NB < 4 ? NB : 4;                  /* blocks of inputs staged a time */
    static constexpr int XS = 32 * XB + 4;                      /* floats of an input row there   */
    static constexpr int WAVE = 2 * 16 * RS;                    /* LDS bytes of a wave's rows     */
};
static_assert(ChFmt<14>::UNITS * 16 <= ChFmt<14>::RS, "whole units in an LDS row");

/* A lane's quarter of a 32-block (the words it trades) and the block's scales. */
template <int TYPE>
struct ChRaw {
    static constexpr int N = TYPE == 0 ? 8 : (TYPE == 1 || TYPE == 14 ? 4 : (TYPE == 8 ? 2 : 1));
    uint32_t q[N];
    uint32_t s, s2;
};

/* Global reads at the rows' alignment (2 bytes for Q8_0, Q4_0 and Q6_K blocks). */
typedef uint32_t u32x4_a2 __attribute__((ext_vector_type(4), aligned(2)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

/* Lane group g's quarter of block b (a constant) of the staged row at p. */
template <int TYPE>
__device__ __forceinline__ void ch_read(const uint8_t *p, int b, int g, ChRaw<TYPE> &r)
{
    if constexpr (TYPE == 0) {
        const u32x4 v0 = *(const u32x4 *)(p + 128 * b + 16 * g), v1 = *(const u32x4 *)(p + 128 * b + 16 * g + 64);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            r.q[i] = v0[i];
            r.q[4 + i] = v1[i];
        }
    } else if constexpr (TYPE == 1) {
        const u32x2 v0 = *(const u32x2 *)(p + 64 * b + 8 * g), v1 = *(const u32x2 *)(p + 64 * b + 8 * g + 32);
        r.q[0] = v0.x;
        r.q[1] = v0.y;
        r.q[2] = v1.x;
        r.q[3] = v1.y;
    } else if constexpr (TYPE == 8) {
        /* even blocks' codes sit 2 bytes past a word: aligned words and a byte shift (LDS reads
         * off their alignment are several times slower) */
        const uint32_t *w = (const uint32_t *)(p + 34 * b + 8 * g + ((b & 1) ? 2 : 0));
        if (b & 1) {
            r.q[0] = w[0];
            r.q[1] = w[1];
        } else {
            r.q[0] = __builtin_amdgcn_alignbyte(w[1], w[0], 2);
            r.q[1] = __builtin_amdgcn_alignbyte(w[2], w[1], 2);
        }
        r.s = *(const uint16_t *)(p + 34 * b);
    } else if constexpr (TYPE == 14) {
        const int hf = (b & 7) >> 2, gb = b & 3;
        const u32x2 lo = *(const u32x2 *)(p + 64 * hf + 32 * (gb & 1) + 8 * g);
        const u32x2 hi = *(const u32x2 *)(p + 128 + 32 * hf + 8 * g);
        r.q[0] = lo.x;
        r.q[1] = lo.y;
        r.q[2] = hi.x;
        r.q[3] = hi.y;
        r.s = *(const uint16_t *)(p + 208);
        r.s2 = *(const uint16_t *)(p + 192 + 8 * hf + 2 * gb);
    } else if constexpr (TYPE == 3) {
        r.s = *(const uint32_t *)(p + 20 * b);
        r.q[0] = *(const uint32_t *)(p + 20 * b + 4 * g + 4);
    } else {
        r.s = *(const uint16_t *)(p + 18 * b);
        const uint32_t *w = (const uint32_t *)(p + 18 * b + 4 * g + ((b & 1) ? 2 : 0));
        r.q[0] = (b & 1) ? w[0] : __builtin_amdgcn_alignbyte(w[1], w[0], 2);
    }
}

/* Lanes 32-63 of x trade with lanes 0-31 of y (32), odd 16-lane rows of x with even ones of y (16). */
__device__ __forceinline__ void swap32(uint32_t &x, uint32_t &y)
{
    const auto r = __builtin_amdgcn_permlane32_swap(x, y, false, false);
    x = r[0];
    y = r[1];
}
__device__ __forceinline__ void swap16(uint32_t &x, uint32_t &y)
{
    const auto r = __builtin_amdgcn_permlane16_swap(x, y, false, false);
    x = r[0];
    y = r[1];
}

/* Byte t of the words a, b of the four lanes of a row (groups s = 0..3) into the lane of group t:
 * a's of s = 0, 2 and b's of s = 0, 2 into a; those of s = 1, 3 into b. */
__device__ __forceinline__ void trade_bytes(uint32_t &a, uint32_t &b)
{
    uint32_t x = __builtin_amdgcn_perm(b, a, 0x05040100u), y = __builtin_amdgcn_perm(b, a, 0x07060302u);
    swap32(x, y);                             /* x from s < 2, y from s >= 2, for groups of one half */
    a = __builtin_amdgcn_perm(y, x, 0x06020400u);
    b = __builtin_amdgcn_perm(y, x, 0x07030501u);
    swap16(a, b);
}

/* Elements 4j + g of the block, j = 0..7, of lane group g as qms_dequant_row forms them. */
template <int TYPE>
__device__ __forceinline__ void ch_vals(const ChRaw<TYPE> &r, int b, float (&v)[8])
{
    if constexpr (TYPE == 0) {
#pragma unroll
        for (int k = 0; k < 2; k++) {
            uint32_t q0 = r.q[4 * k], q1 = r.q[4 * k + 1], q2 = r.q[4 * k + 2], q3 = r.q[4 * k + 3];
            swap32(q0, q2);                   /* q0, q1 from s < 2; q2, q3 from s >= 2              */
            swap32(q1, q3);
            swap16(q0, q1);                   /* q0, q2 from even s; q1, q3 from odd s              */
            swap16(q2, q3);
            v[4 * k] = __uint_as_float(q0);
            v[4 * k + 1] = __uint_as_float(q1);
            v[4 * k + 2] = __uint_as_float(q2);
            v[4 * k + 3] = __uint_as_float(q3);
        }
    } else if constexpr (TYPE == 1) {
#pragma unroll
        for (int k = 0; k < 2; k++) {
            uint32_t x = r.q[2 * k], y = r.q[2 * k + 1];
            swap32(x, y);
            uint32_t u = __builtin_amdgcn_perm(y, x, 0x05040100u), w = __builtin_amdgcn_perm(y, x, 0x07060302u);
            swap16(u, w);                     /* u: s = 0, 2; w: s = 1, 3                            */
            v[4 * k] = h2f(u & 0xffffu);
            v[4 * k + 1] = h2f(w & 0xffffu);
            v[4 * k + 2] = h2f(u >> 16);
            v[4 * k + 3] = h2f(w >> 16);
        }
    } else if constexpr (TYPE == 8) {
        uint32_t u = r.q[0], w = r.q[1];
        trade_bytes(u, w);                    /* u: words 0, 4, 1, 5 of the block; w: 2, 6, 3, 7     */
        const float d = h2f(r.s & 0xffffu);
        auto val = [d](uint32_t x, int k) { return (float)(int8_t)((x >> (8 * k)) & 0xffu) * d; };
        v[0] = val(u, 0);
        v[4] = val(u, 1);
        v[1] = val(u, 2);
        v[5] = val(u, 3);
        v[2] = val(w, 0);
        v[6] = val(w, 1);
        v[3] = val(w, 2);
        v[7] = val(w, 3);
    } else if constexpr (TYPE == 14) {
        uint32_t u = r.q[0], w = r.q[1], hu = r.q[2], hw = r.q[3];
        trade_bytes(u, w);
        trade_bytes(hu, hw);
        const int gb = b & 3, ns = gb & 2 ? 4 : 0, hs = 2 * gb;
        const uint32_t cu = ((u >> ns) & 0x0f0f0f0fu) | (((hu >> hs) & 0x03030303u) << 4);
        const uint32_t cw = ((w >> ns) & 0x0f0f0f0fu) | (((hw >> hs) & 0x03030303u) << 4);
        const float d = h2f(r.s & 0xffffu), d0 = d * (float)(int8_t)(r.s2 & 0xff), d1 = d * (float)(int8_t)(r.s2 >> 8);
        auto val = [](uint32_t x, int k, float dd) { return dd * (float)((int)((x >> (8 * k)) & 0xffu) - 32); };
        v[0] = val(cu, 0, d0);
        v[4] = val(cu, 1, d1);
        v[1] = val(cu, 2, d0);
        v[5] = val(cu, 3, d1);
        v[2] = val(cw, 0, d0);
        v[6] = val(cw, 1, d1);
        v[3] = val(cw, 2, d0);
        v[7] = val(cw, 3, d1);
    } else {
        /* a code word of each lane: low nibbles elements 4s + t, high nibbles 16 + 4s + t */
        uint32_t x = r.q[0], y = r.q[0] >> 16;
        swap32(x, y);
        uint32_t u = __builtin_amdgcn_perm(y, x, 0x0c0c0400u), w = __builtin_amdgcn_perm(y, x, 0x0c0c0501u);
        swap16(u, w);                         /* u: s = 0, 2; w: s = 1, 3                            */
        const float d = h2f(r.s & 0xffffu), m = TYPE == 3 ? h2f(r.s >> 16) : 0.0f;
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const uint32_t c = (((j & 1) ? w : u) >> (8 * ((j >> 1) & 1) + (j >= 4 ? 4 : 0))) & 15u;
            if constexpr (TYPE == 3) v[j] = __builtin_fmaf((float)c, d, m);
            else v[j] = (float)((int)c - 8) * d;
        }
    }
}

/* LDS bytes: the four waves' row buffers, then two stages of 16 NC input rows or T rows of C. */
template <int TYPE>
size_t ch_lds(int NC) { return 4 * (size_t)ChFmt<TYPE>::WAVE + 2 * (size_t)(16 * NC * ChFmt<TYPE>::XS) * 4; }
template <int TYPE>
size_t ch_lds_res(int T, int C) { return 4 * (size_t)ChFmt<TYPE>::WAVE + chain_rows_lds(T, C); }

/* The chains of a wave's 16 rows over nblk 32-blocks: row i (clamped to rows - 1) at wb + i * rb, wb
 * wave-uniform; acc[n] takes row 4 (lane / 16) + v, input row 16 n + lane % 16. Not RES: thread t
 * stages the input rows xr[n] for t / 16 + 16 n at xsm. RES: the block has staged its input rows
 * (chain_rows_lds), and xl is the lane's row there. Every wave passes the same barriers; all
 * LDS reads are done at the end except other waves' (of their own rows, or of RES inputs). */
template <int TYPE, int NC, bool RES>
__device__ __forceinline__ void chain_tile(uint8_t *wsm, float *xsm, const uint8_t *wb, uint32_t rb, int rows,
                                           const float *const (&xr)[NC], const float *xl, int nblk, f32x4 (&acc)[NC])
{
    static_assert(!RES || NC == 1, "staged whole: one instruction's input rows");
    using F = ChFmt<TYPE>;
    constexpr int R = RES ? 2 : 1;            /* chunks in flight in registers (four: no faster) */
    constexpr int NB = F::NB, XB = F::XB, XBUF = 16 * NC * F::XS, NX = RES ? 1 : NC * XB / 2;
    const int tid = threadIdx.x, lane = tid & 63, i = lane & 15, g = lane >> 4;
    const int nch = (nblk + NB - 1) / NB, nfull = nblk / NB;
    /* weight units 64 q + lane: (row, 16-byte unit); units past the row's end read its last bytes'
     * neighbours (at most 15 bytes past the tensor, inside its allocation's padding) */
    uint32_t vo[F::NL], vu[F::NL], ldo[F::NL];
#pragma unroll
    for (int q = 0; q < F::NL; q++) {
        const int n = min(64 * q + lane, 16 * F::UNITS - 1), row = n / F::UNITS, u = n - row * F::UNITS;
        vo[q] = (uint32_t)min(row, rows - 1) * rb;
        vu[q] = 16u * (uint32_t)u;
        ldo[q] = (uint32_t)(row * F::RS + 16 * u);
    }
    u32x4 wv[R][F::NL];
    auto load_w = [&](int c, int k) {
        /* no condition, so that each wait covers one chunk's loads and not all in flight: past the
         * last chunk every lane reads the first row's first bytes */
        const uint32_t cb = (uint32_t)c * F::BYTES, mask = c < nch ? ~0u : 0u;
#pragma unroll
        for (int q = 0; q < F::NL; q++)
            wv[k][q] = *(const u32x4_a2 *)(wb + ((vo[q] + min(cb + vu[q], rb - 2u)) & mask));
    };
    auto store_w = [&](int c, int k) {
#pragma unroll
        for (int q = 0; q < F::NL; q++) *(u32x4 *)(wsm + (c & 1) * (16 * F::RS) + ldo[q]) = wv[k][q];
        /* the wave's LDS accesses run in order; keep the compiler to it */
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    };
    /* inputs: float4 p of thread tid covers row tid / 16 + 16 n, float4 16 m + tid % 16 of the
     * stage's 8 XB */
    f32x4 xv[NX];
    auto load_x = [&](int st) {
        if constexpr (!RES)
#pragma unroll
            for (int n = 0; n < NC; n++)
#pragma unroll
                for (int m = 0; m < XB / 2; m++) {
                    const int f = 16 * m + (tid & 15);
                    const int e = 32 * min(XB * st + (f >> 3), nblk - 1) + 4 * (f & 7);
                    xv[n * (XB / 2) + m] = *(const f32x4 *)(xr[n] + e);
                }
    };
    auto store_x = [&](int st) {
        if constexpr (!RES)
#pragma unroll
            for (int n = 0; n < NC; n++)
#pragma unroll
                for (int m = 0; m < XB / 2; m++) {
                    const int f = 16 * m + (tid & 15);
                    float *d = xsm + (st & 1) * XBUF + (16 * n + (tid >> 4)) * F::XS + 32 * (f >> 3) + (f & 7);
#pragma unroll
                    for (int k = 0; k < 4; k++) d[8 * k] = xv[n * (XB / 2) + m][k];
                }
    };
    f32x4 b0[NC][2], b1[NC][2];
    auto read_b = [&](int st, int k, f32x4 (&b)[NC][2]) {
#pragma unroll
        for (int n = 0; n < NC; n++)
#pragma unroll
            for (int q = 0; q < 2; q++)
                b[n][q] = *(const f32x4 *)(RES ? xl + chain_row_read(XB * st + k, g, q)
                                               : xsm + (st & 1) * XBUF + (16 * n + i) * F::XS + 32 * k + 8 * g + 4 * q);
    };
    float a[8];
#pragma unroll
    for (int n = 0; n < NC; n++) acc[n] = f32x4{ 0.0f, 0.0f, 0.0f, 0.0f };
    load_x(0);
#pragma unroll
    for (int k = 0; k < R; k++) load_w(k, k);
    store_x(0);
    store_w(0, 0);
    load_x(1);
    load_w(R, 0);
    ChRaw<TYPE> r1;                           /* the next block's words                           */
    ch_read<TYPE>(wsm + i * F::RS, 0, g, r1);
    ch_vals<TYPE>(r1, 0, a);
    ch_read<TYPE>(wsm + i * F::RS, 1, g, r1);
    if constexpr (!RES) mx_lds_barrier();
    if (RES) read_b(0, 0, b0);
    /* chunk c, whose bytes are in LDS, with block 0's weights in a: the next chunk's bytes go to the
     * other buffer first, and every block's inputs are read, and the weights of the one after it, while
     * the previous block's instructions run */
    auto chunk = [&](int c, int k, auto full_c) {
        constexpr bool FULL = decltype(full_c)::value;
        store_w(c + 1, k);
        load_w(c + 1 + R, k);
        __builtin_amdgcn_sched_barrier(0);
        const uint8_t *wp = wsm + (c & 1) * (16 * F::RS) + i * F::RS, *wn = wsm + ((c + 1) & 1) * (16 * F::RS) + i * F::RS;
#pragma unroll
        for (int h = 0; h < NB / XB; h++) {
            const int st = c * (NB / XB) + h;
            if (!FULL && XB * st >= nblk) break;
            store_x(st + 1);
            load_x(st + 2);
            if constexpr (!RES) read_b(st, 0, b0);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int kk = 0; kk < XB; kk++) {
                if (!FULL && XB * st + kk >= nblk) break;
                const int b = XB * h + kk;
                ChRaw<TYPE> r2;
                if (b + 2 < NB) ch_read<TYPE>(wp, b + 2, g, r2);
                else ch_read<TYPE>(wn, b + 2 - NB, g, r2);
                if (RES || kk + 1 < XB) {
                    if (kk & 1) read_b(st, kk + 1, b0);
                    else read_b(st, kk + 1, b1);
                }
                float an[8];
                ch_vals<TYPE>(r1, (b + 1) % NB, an);
#pragma unroll
                for (int j = 0; j < 8; j++)
#pragma unroll
                    for (int n = 0; n < NC; n++)
                        acc[n] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[j], (kk & 1 ? b1 : b0)[n][j >> 2][j & 3], acc[n],
                                                                      0, 0, 0);
#pragma unroll
                for (int j = 0; j < 8; j++) a[j] = an[j];
                r1 = r2;
                /* the vector instructions of the next block's weights between the matrix ones, whose
                 * chain otherwise stalls the wave 32 cycles at each */
                __builtin_amdgcn_sched_group_barrier(0x100, 16, 0);
#pragma unroll
                for (int j = 0; j < 8; j++) {
                    __builtin_amdgcn_sched_group_barrier(0x008, NC, 0);
                    __builtin_amdgcn_sched_group_barrier(0x002, 5, 0);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            if constexpr (!RES) mx_lds_barrier();
        }
    };
    int c = 0;
    for (; c + R <= nfull; c += R)
#pragma unroll
        for (int k = 0; k < R; k++) chunk(c + k, (k + 1) % R, std::true_type{});
#pragma unroll
    for (int k = 0; k < R; k++) {
        if (c + k < nfull) chunk(c + k, (k + 1) % R, std::true_type{});
        else if (c + k < nch) chunk(c + k, (k + 1) % R, std::false_type{});
    }
}

/* chain_tile for a block of nt input rows: the second sixteen's work only where there are any. */
template <int TYPE, int NC, bool RES>
__device__ __forceinline__ void chain_rows_of(uint8_t *smem, const uint8_t *wb, uint64_t rb, int rows,
                                              const float *const (&xr)[NC], const float *xl, int nblk, int nt,
                                              f32x4 (&acc)[NC])
{
    uint8_t *wsm = smem + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) * ChFmt<TYPE>::WAVE;
    float *xsm = (float *)(smem + 4 * ChFmt<TYPE>::WAVE);
    if constexpr (NC == 2) {
        if (nt <= 16) {
            const float *const x1[1] = { xr[0] };
            f32x4 one[1];
            chain_tile<TYPE, 1, RES>(wsm, xsm, wb, (uint32_t)rb, rows, x1, xl, nblk, one);
            acc[0] = one[0];
            acc[1] = f32x4{ 0.0f, 0.0f, 0.0f, 0.0f };
            return;
        }
    }
    chain_tile<TYPE, NC, RES>(wsm, xsm, wb, (uint32_t)rb, rows, xr, xl, nblk, acc);
}

/* Input rows staged whole, as [row][block][g][8] at chain_row_floats(C) per row; src(r) is row r. */
template <class Src>
__device__ __forceinline__ void chain_stage(float *xsm, int rows, int C, Src src)
{
    const int q4 = C >> 2;
    for (int k = threadIdx.x; k < rows * q4; k += 256) {
        const int r = k / q4, q = k - r * q4;
        const f32x4 v = *(const f32x4 *)(src(r) + 4 * q);
        float *d = xsm + r * chain_row_floats(C) + 32 * (q >> 3) + (q & 7);
#pragma unroll
        for (int j = 0; j < 4; j++) d[8 * j] = v[j];
    }
    __syncthreads();
}

/* Rows of one expert tensor (or of gate and up) for the slots of a slot tile. */
struct ChainArgs {
    const uint8_t *w, *w2;        /* the tensor; PAIR: gate and up                          */
    uint64_t rb, eb, rb2, eb2;
    int rows, cols, by_token;     /* by_token: slot s reads row slot_t[s] of x, else row s  */
    const float *x;
    float *y;                     /* y[slot * y_stride + row]; PAIR: act [slot][rows]       */
    int y_stride;
    float *gu;                    /* PAIR: [slot][2 rows] gate then up rows, or NULL        */
    Scratch S;
};

/* PAIR: 32 gate rows and the same 32 up rows, a = silu(g) * u (src/model.c:1024) in the block. */
template <int TYPE, int NC, bool PAIR, bool RES>
__global__ __launch_bounds__(256) void chain_rows_kernel(ChainArgs a)
{
    extern __shared__ __align__(16) uint8_t chsm[];
    const int tile = (int)(blockIdx.z * gridDim.y + blockIdx.y);
    if (tile >= a.S.meta[1]) return;
    const int4 tl = a.S.tiles[tile];
    const int e = tl.x, s0 = tl.y, ns = tl.z - tl.y;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int R0 = (int)blockIdx.x * (PAIR ? 32 : 64);
    /* PAIR: waves 0, 1 gate rows, waves 2, 3 the same up rows */
    const bool second = PAIR && wave >= 2;
    const int rw = R0 + 16 * (PAIR ? wave & 1 : wave), rbase = min(rw, a.rows - 1);
    const uint64_t rb = second ? a.rb2 : a.rb;
    const uint8_t *wb = (second ? a.w2 + (size_t)e * a.eb2 : a.w + (size_t)e * a.eb) + (size_t)rbase * rb;
    auto src = [&](int r) {
        const int s = s0 + min(r, ns - 1);
        return a.x + (size_t)(a.by_token ? a.S.slot_t[s] : s) * a.cols;
    };
    const float *xr[NC], *xl = nullptr;
    if constexpr (RES) {
        float *xsm = (float *)(chsm + 4 * ChFmt<TYPE>::WAVE);
        chain_stage(xsm, ns, a.cols, src);
        xl = xsm + min(lane & 15, ns - 1) * chain_row_floats(a.cols);
        xr[0] = nullptr;
    } else {
#pragma unroll
        for (int n = 0; n < NC; n++) xr[n] = src(16 * n + (tid >> 4));
    }
    f32x4 acc[NC];
    chain_rows_of<TYPE, NC, RES>(chsm, wb, rb, a.rows - rbase, xr, xl, a.cols >> 5, ns, acc);
    const int r = 16 * wave + 4 * (lane >> 4), sl = lane & 15;
    if constexpr (PAIR) {
        constexpr int RS = 16 * NC + 1;
        float *res = (float *)chsm;
        __syncthreads();                          /* every wave is past its LDS reads */
#pragma unroll
        for (int n = 0; n < NC; n++)
#pragma unroll
            for (int v = 0; v < 4; v++) res[(r + v) * RS + 16 * n + sl] = acc[n][v];
        __syncthreads();
        for (int k = tid; k < 32 * ns; k += 256) {
            const int f = k & 31, s = k >> 5;
            if (R0 + f >= a.rows) continue;
            const float gv = res[f * RS + s], uv = res[(32 + f) * RS + s];
            a.y[(size_t)(s0 + s) * a.y_stride + R0 + f] = silu_ref(gv) * uv;
            if (a.gu) {
                float *gu = a.gu + (size_t)(s0 + s) * 2 * a.rows + R0 + f;
                gu[0] = gv;
                gu[a.rows] = uv;
            }
        }
    } else {
#pragma unroll
        for (int n = 0; n < NC; n++)
#pragma unroll
            for (int v = 0; v < 4; v++)
                if (16 * n + sl < ns && R0 + r + v < a.rows)
                    a.y[(size_t)(s0 + 16 * n + sl) * a.y_stride + R0 + r + v] = acc[n][v];
    }
}

/* matmul_exact for up to kDenseMats resident matrices of one type against T input rows: block
 * x takes 64 rows of the matrix whose block range holds it, (y, z) the input rows in 16 NC's. */
template <int TYPE, int NC, bool RES>
__global__ __launch_bounds__(256) void chain_dense_kernel(DenseArgs a)
{
    extern __shared__ __align__(16) uint8_t chsm[];
    int mi = 0;
#pragma unroll
    for (int i = 1; i < kDenseMats; i++)
        if (i < a.nm && (int)blockIdx.x >= a.m[i].first_block) mi = i;
    const DenseMat M = a.m[mi];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int R0 = ((int)blockIdx.x - M.first_block) * kChRows;
    const int t0 = ((int)blockIdx.z * (int)gridDim.y + (int)blockIdx.y) * 16 * NC, nt = min(16 * NC, a.T - t0);
    if (nt <= 0) return;
    const int rw = R0 + 16 * wave, rbase = min(rw, M.rows - 1);
    const uint8_t *wb = M.w + (size_t)rbase * a.rb;
    auto src = [&](int r) { return a.x + (size_t)(t0 + min(r, nt - 1)) * a.C; };
    const float *xr[NC], *xl = nullptr;
    if constexpr (RES) {
        float *xsm = (float *)(chsm + 4 * ChFmt<TYPE>::WAVE);
        chain_stage(xsm, nt, a.C, src);
        xl = xsm + min(lane & 15, nt - 1) * chain_row_floats(a.C);
        xr[0] = nullptr;
    } else {
#pragma unroll
        for (int n = 0; n < NC; n++) xr[n] = src(16 * n + (tid >> 4));
    }
    f32x4 acc[NC];
    chain_rows_of<TYPE, NC, RES>(chsm, wb, a.rb, M.rows - rbase, xr, xl, a.C >> 5, nt, acc);
    const int r = 16 * wave + 4 * (lane >> 4), sl = lane & 15;
#pragma unroll
    for (int n = 0; n < NC; n++)
#pragma unroll
        for (int v = 0; v < 4; v++)
            if (16 * n + sl < nt && R0 + r + v < M.rows)
                M.y[(size_t)(t0 + 16 * n + sl) * M.rows + R0 + r + v] = acc[n][v];
}

/* f(type tag) for a GGUF tensor type the chains take; false for any other. */
template <int T>
struct TypeTag {
    static constexpr int value = T;
};
template <class F>
bool with_type(int type, F f)
{
    switch (type) {
    case 0: f(TypeTag<0>{}); return true;
    case 1: f(TypeTag<1>{}); return true;
    case 2: f(TypeTag<2>{}); return true;
    case 3: f(TypeTag<3>{}); return true;
    case 8: f(TypeTag<8>{}); return true;
    case 14: f(TypeTag<14>{}); return true;
    default: return false;
    }
}

/* Tiles over y and z: a grid's y ends at 65535, and 32,768 tokens of 64 experts make more. */
dim3 chain_grid(int blocks, int tiles)
{
    const int ty = tiles < 32768 ? tiles : 32768;
    return dim3(blocks, ty, (tiles + ty - 1) / ty);
}

}  // namespace

hipError_t launch_chain_rows(const char *name, const ChainRows &m, const ChainRows *up, const Scratch &S, int T,
                             int max_tiles, float *gu, hipStream_t st)
{
    ChainArgs a;
    a.w = m.w;
    a.rb = m.rb;
    a.eb = m.eb;
    a.w2 = up ? up->w : nullptr;
    a.rb2 = up ? up->rb : 0;
    a.eb2 = up ? up->eb : 0;
    a.rows = m.rows;
    a.cols = m.cols;
    a.by_token = m.by_token;
    a.x = m.x;
    a.y = m.y;
    a.y_stride = m.y_stride;
    a.gu = gu;
    a.S = S;
    const dim3 grid = chain_grid((m.rows + (up ? 31 : 63)) / (up ? 32 : 64), max_tiles), block(256);
    const bool ok = with_type(m.type, [&](auto ty) {
        constexpr int TY = decltype(ty)::value;
        /* LDS of the inputs whole, or of stages; gate/up's results take less than either */
        static_assert(64 * 33 * 4 <= 4 * ChFmt<TY>::WAVE, "results of 32 slots fit in the row buffers");
        const size_t whole = ch_lds_res<TY>(T, m.cols);
        /* an expert's slots are distinct tokens: up to 16 tokens every slot tile fits one
         * instruction's columns, and its input rows LDS where T of them do. Grids of experts are
         * several times the CUs, and a block that takes more than half a CU's LDS loses more than
         * whole inputs gain (us a layer, whole / in stages: 30B, Q4_0 with Q8_0 down, 16 tokens
         * 209 / 190; Q8_0 6 tokens 141 / 132; 235B --exact, Q4_0, 4 tokens 327 / 293; below the line
         * 126 / 137 at one token) */
        const bool res = T <= 16 && (size_t)T * m.cols <= kChResFloats && whole <= kChResLds;
        if (up) {
            if (res) QLAUNCH(name, (chain_rows_kernel<TY, 1, true, true>), grid, block, whole, st, a);
            else if (T <= 16) QLAUNCH(name, (chain_rows_kernel<TY, 1, true, false>), grid, block, ch_lds<TY>(1), st, a);
            else QLAUNCH(name, (chain_rows_kernel<TY, 2, true, false>), grid, block, ch_lds<TY>(2), st, a);
        } else {
            if (res) QLAUNCH(name, (chain_rows_kernel<TY, 1, false, true>), grid, block, whole, st, a);
            else if (T <= 16) QLAUNCH(name, (chain_rows_kernel<TY, 1, false, false>), grid, block, ch_lds<TY>(1), st, a);
            else QLAUNCH(name, (chain_rows_kernel<TY, 2, false, false>), grid, block, ch_lds<TY>(2), st, a);
        }
    });
    return ok ? hipGetLastError() : hipErrorInvalidValue;
}

hipError_t launch_dense_exact(const DenseArgs &args, int type, hipStream_t st)
{
    DenseArgs a = args;
    int nblk = 0;
    for (int i = 0; i < a.nm; i++) {
        a.m[i].first_block = nblk;
        nblk += (a.m[i].rows + kChRows - 1) / kChRows;
    }
    const dim3 grid = chain_grid(nblk, (a.T + 31) / 32);
    const bool ok = with_type(type, [&](auto tag) {
        constexpr int TY = decltype(tag)::value;
        const size_t whole = ch_lds_res<TY>(a.T, a.C);
        if (a.T <= 16 && (size_t)a.T * a.C <= kChResFloats)
            QLAUNCH("dense", (chain_dense_kernel<TY, 1, true>), dim3(nblk), dim3(256), whole, st, a);
        else if (a.T <= 16) QLAUNCH("dense", (chain_dense_kernel<TY, 1, false>), dim3(nblk), dim3(256), ch_lds<TY>(1), st, a);
        else QLAUNCH("dense", (chain_dense_kernel<TY, 2, false>), grid, dim3(256), ch_lds<TY>(2), st, a);
    });
    return ok ? hipGetLastError() : hipErrorInvalidValue;
}

}  // namespace qmsg
