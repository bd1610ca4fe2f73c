/* qmsg_internal.h - shapes and device pointers shared by the host API and the kernels. */
#ifndef QMSG_INTERNAL_H
#define QMSG_INTERNAL_H

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace qmsg {

/* QmsQ8 (src/kernels.h:7-12): the reference's 44-byte int8 activation block. */
struct Q8 {
    float d;
    float ds;
    int16_t s16[2];
    int8_t q[32];
};
static_assert(sizeof(Q8) == 44, "QmsQ8 is 44 bytes");

/* Kernel-side copy of the same blocks, grouped by pairs of 32-blocks (b even, b+1) so one
 * 16-byte LDS read gives a lane both of its code dwords for two blocks. 96 bytes per pair:
 *   [16p .. 16p+15]  for lane p = 0..3: q[4p..4p+3] of b, q[16+4p..] of b,
 *                                        q[4p..4p+3] of b+1, q[16+4p..] of b+1
 *   [64 .. 79]       d(b), ds(b), d(b+1), ds(b+1)
 *   [80 .. 87]       s16 pair of b, s16 pair of b+1 (low half = s16[0])
 *   [88 .. 95]       zero */
constexpr int kPairBytes = 96;

/* Optional per-dispatch timing. While a hook is installed on the calling thread, every kernel
 * launch of the library asks it for an event pair and launches through hipExtLaunchKernel,
 * which stamps the dispatch's own start and end into the events (no marker packets between
 * kernels). `kernel` is the launch's short name: route, select, dispatch, gateup, down,
 * combine, copy. */
struct LaunchTimer {
    void *ctx;
    void (*events)(void *ctx, const char *kernel, hipEvent_t *start, hipEvent_t *stop);
};
extern thread_local const LaunchTimer *g_launch_timer;

/* Static shape limits of the kernels. */
constexpr int kMaxExperts = 256;

/* Slots (tokens of one expert) per slot tile of the batch kernels (dispatch's tile list). */
constexpr int kTileN = 32;
/* Bytes of one activation record of the MFMA kernels (one int8 block as f16 codes, its scales
 * and the MFMA accumulator inputs). */
constexpr int kMxRec = 128;

/* The default path takes the MFMA kernels for gate/up once a batch averages kMxAutoQuarters / 4
 * slots per active expert, and for down from kMxDownMinSlotsQ4 slots (Q4_0 / Q4_1 rows, and Q6_K rows
 * of an odd number of super-blocks below kMxDownOddCols columns) or kMxDownMinSlotsQ6 (other Q6_K
 * rows). Gate/up at the 235B shape, MFMA against the row kernels with the records each needs (us):
 * 132.2 / 130.1 at 16 tokens, 114.2 / 107.1 at 12, and from 20 tokens (1.25 slots per expert) 149.6 /
 * 154.8. Down after row-kernel gate/up, us of the layer, MFMA / row kernels: 235B Q4_0 89 / 86 at 4
 * tokens, 118 / 119 at 6, 141 / 144 at 8, 217 / 228 at 16, 30B 56.2 / 53.7 at 6, 62.5 / 61.1 at 8, 71.3
 * / 72.3 at 10 (Q4_1 the same within 2); 235B Q6_K 72 / 69 at 2, 93 / 95 at 3, 111 / 113 at 4, 129 / 153
 * at 5. Odd rows: 1280 columns under 4096 rows 67 / 70 at 2, 101 / 118 at 4; 768 under 2048 (30B)
 * 55.3 / 55.5 at 4, 62.7 / 59.8 at 5, 67.8 / 66.9 at 7, 72.5 / 72.0 at 8, 82 / 85 at 10; 768 under 1024
 * 42.2 / 40.3 at 4, 52.2 / 51.6 at 8. */
constexpr int kMxAutoQuarters = 5;
/* Q6_K gate/up (its MFMA kernel unpacks 6-bit codes): from 2.5 slots per expert (streaming /
 * MFMA us: 442 / 487 at 32 tokens, 618 / 435 at 48) */
constexpr int kMxAutoQuartersQ6 = 10;
constexpr int kMxDownMinSlotsQ4 = 64;
constexpr int kMxDownMinSlotsQ6 = 32;
constexpr int kMxDownOddCols = 1024;
inline bool mx_auto(int T, int K, int X, int gate_type)
{
    const long NS = (long)T * K, act = X < NS ? X : NS;
    return 4 * NS >= (long)(gate_type == 14 ? kMxAutoQuartersQ6 : kMxAutoQuarters) * act;
}
inline bool mx_auto_down(int T, int K, int F, int down_type)
{
    const bool late = down_type != 14 || (F % 512 != 0 && F < kMxDownOddCols);
    return (long)T * K >= (late ? kMxDownMinSlotsQ4 : kMxDownMinSlotsQ6);
}

/* One-token batches (n_used <= 8) are routed inside the gate/up kernel instead of by a
 * separate select launch. */
inline int use_small_route(int T, int K) { return T == 1 && K <= 8; }

/* Per-layer device weights: the GGUF bytes, unchanged, in one allocation per tensor. */
struct LayerDev {
    const float *router;    /* [X][E] */
    const uint8_t *gate;    /* [X][F] rows of gate_rb bytes */
    const uint8_t *up;      /* [X][F] rows of up_rb bytes   */
    const uint8_t *down;    /* [X][E] rows of down_rb bytes */
    int gate_type, up_type, down_type;
    uint64_t gate_rb, up_rb, down_rb;
    uint64_t gate_eb, up_eb, down_eb;
};

/* Device scratch of a context, sized for max_tokens. */
struct Scratch {
    float *logits;      /* [Tm][X]             */
    int32_t *sel;       /* [Tm*K]              */
    float *wt;          /* [Tm*K]              */
    int32_t *slot_t;    /* [Tm*K]              */
    int32_t *slot_of;   /* [Tm*K]              */
    int32_t *start;     /* [X+1]               */
    int32_t *active;    /* [X]                 */
    int4 *work;         /* [X] per active expert: {expert, first slot, end slot, 0}; expert -1 after */
    int4 *tiles;        /* [X + Tm*K/kTileN + 1] slot tiles of the MFMA kernels: {expert, first, end, 0} */
    int32_t *meta;      /* [0] n_active, [1] number of slot tiles */
    Q8 *xq;             /* [Tm][E/32]          */
    uint8_t *xqk;       /* [Tm][E/64][96]      */
    float *gu;          /* [Tm*K][2F]          */
    float *act;         /* [Tm*K][F]           */
    Q8 *aq;             /* [Tm*K][F/32]        */
    uint8_t *aqk;       /* [Tm*K][F/64][96]    */
    float *dn;          /* [Tm*K][E]           */
    uint8_t *mxx;       /* [Tm][E/32][kMxRec] MFMA records of the layer input */
    uint8_t *mxa;       /* [Tm*K][F/32][kMxRec] MFMA records of the activations */
    uint64_t *mxflag;   /* [2] the epoch of the last call whose input (0) / activation (1) records
                         * hold a d_x outside the MFMA kernels' scaled range */
    uint64_t epoch;     /* this call's epoch (unique per layer call in the process) */
};

struct Shape {
    int E, X, K, F;
};

/* Dense (trunk) matrices of one qms_matmul_n call: same type and cols, at most kDenseMats. */
constexpr int kDenseMats = 4;
struct DenseMat {
    const uint8_t *w;       /* rows of rb bytes (GGUF layout) */
    float *y;               /* [T][rows]                      */
    int rows;
    int first_block;        /* set by the launcher            */
};
struct DenseArgs {
    DenseMat m[kDenseMats];
    int nm;
    uint64_t rb;
    int C, T;
    const float *x;         /* [T][C] input rows (16-byte aligned) */
    const uint8_t *xqk;     /* [T][C/64] pair records, or NULL: the kernel quantises x */
};

/* Dense row kernels: batches of at least this many rows are quantised once by a separate launch,
 * smaller ones inside every block. */
constexpr int kDenseQuantT = 8;
/* Rows of more columns can be too long for the row kernels' LDS at several tokens (Q6_K above 16,384,
 * Q4_0 / Q4_1 above 25,600): there the MFMA kernels stay first. */
constexpr int kDenseRowCols = 16384;

/* Whether a call's matrices take the MFMA kernels: rows in whole staged chunks that the LDS DMA can
 * read (Q6_K: 4-byte aligned), a block's rows in each matrix and their bytes in the 31 bits of its
 * offsets (128 rows of under 2^24 bytes), and enough tokens. From 9 tokens always: the row kernels
 * then take another pass, and the smallest lose nothing (us at 9 tokens, row / MFMA kernels, records
 * included: Q4_0 128x256 6.9 / 6.9, 512x1024 12.0 / 9.6, 4096x4096 29.5 / 21.1; Q6_K 130x512 13.2 / 9.1,
 * 512x2048 29.4 / 22.1). At 5-8 tokens by rows:
 * up to 4096 the row kernels' 16-row blocks fit the CUs once and win (5 tokens: Q4_0 4096x4096 18.6 /
 * 20.9, 4096x8192 32.4 / 36.1; Q6_K 28.0 / 38.4, 51 / 72), above it not (Q4_0 6144x4096 23.7 / 21.1,
 * 8192x2048 14.2 / 13.7; Q6_K 6144x4096 53 / 39, 10240x2048 30.4 / 23.9), save small matrices, where
 * the records cost what is gained (Q4_0 6144x1024 8.5 / 9.3; Q6_K 8192x2048 20.2 / 22.8). */
inline bool dense_mx_takes(const DenseArgs &a, int type)
{
    if ((type != 2 && type != 3 && type != 14) || a.C % 256 || (type == 14 && a.rb % 4) || a.rb >= 1u << 24 || a.T > 4 * 65535)
        return false;
    long rows = 0;
    for (int i = 0; i < a.nm; i++) {
        if (a.m[i].rows < 128) return false;
        rows += a.m[i].rows;
    }
    if (a.T > 8) return true;
    if (a.C > kDenseRowCols) return a.T > 4 && rows * a.C >= 1l << 24;
    return a.T > 4 && rows > 4096 && rows * a.C >= (type == 14 ? 5l << 22 : 1l << 24);
}

/* Widths of the chunked row kernels (others: the direct-read kernel), and whether those read pair
 * records from the record buffer (else every block quantises the rows it reads). */
inline bool dense_chunked(int type, int C) { return type == 14 ? C % 2048 == 0 : C % 256 == 0; }
inline bool dense_pairs_taken(int type, int C, int T) { return type != 0 && dense_chunked(type, C) && T >= kDenseQuantT; }

/* Launchers (qmsg_kernels.hip). Each returns hipSuccess or the launch error. */
hipError_t launch_route(const Shape &s, const LayerDev &L, const Scratch &S, const float *xn, int T,
                        hipStream_t st);
/* Top-K and dispatch; a one-token batch is left to the Q4_0 gate/up kernel when gateup_routes. */
hipError_t launch_select(const Shape &s, const Scratch &S, int T, int gateup_routes, hipStream_t st);
/* Whether gate and up take the streaming gate/up kernel (launch_gateup_exact): one type, Q4_0,
 * Q4_1, or Q6_K with rows a multiple of 4 bytes long. */
bool gateup_streams(const LayerDev &L);
/* quant_act: batches (not the one-token routing kernel) in blocks of 32 rows that also store
 * the activations' int8 blocks (aq, aqk) for the down kernel. */
hipError_t launch_gateup_exact(const Shape &s, const LayerDev &L, const Scratch &S, int T, int debug, int n_cu,
                               int quant_act, hipStream_t st);
/* The expert products on the matrix cores (order-exact): gate/up, then down and the combine.
 * mx_supported: whether the layer's types and shape fit the MFMA kernels (gate and up of one
 * type: Q4_0, Q4_1 or Q6_K;
 * *down_mx: whether down runs on them too, else on the exact down kernel). */
bool mx_supported(const Shape &s, const LayerDev &L, int *down_mx);
hipError_t launch_experts_mx(const Shape &s, const LayerDev &L, const Scratch &S, float *out, int T, int debug,
                             hipStream_t st);
/* Down alone on the MFMA kernels after a row-kernel gate/up: activation blocks and records from
 * act, the down tiles, the combine (needs *down_mx of mx_supported). */
hipError_t launch_down_mx(const Shape &s, const LayerDev &L, const Scratch &S, float *out, int T, hipStream_t st);
/* Gate/up rows of Q4_1 / Q6_K (or mixed) layers by slot tiles, then the SwiGLU. */
hipError_t launch_gateup_tiles(const Shape &s, const LayerDev &L, const Scratch &S, int T, hipStream_t st);
/* Whether two to four tokens take the small-batch down kernel. */
bool down_small_fits(const Shape &s, const LayerDev &L, int T);
/* Whether one of the exact down kernels (one-token, small-batch, slot tiles) holds this shape
 * in LDS; rows too long for all of them take the MFMA down kernel, which stages them in chunks. */
bool down_exact_fits(const Shape &s, const LayerDev &L, int T);
/* quant: the activations' int8 blocks are formed here (else read from aqk, where gate/up or the
 * MFMA gate/up stored them). */
hipError_t launch_down_exact(const Shape &s, const LayerDev &L, const Scratch &S, float *out, int T, int quant,
                             hipStream_t st);
/* The whole layer slot by slot, as the reference's moe_group_exact (src/model.c:1009-1030): with
 * exact its --exact mode (fp32 dequantised rows, fp32 activations), else each qms_matmul on its
 * int8 path, for shapes off the integer kernels' grid (integer_grid_shape). debug also stores
 * the int8 blocks of the inputs and activations (xq, aq) that the slot kernels keep in LDS. */
hipError_t launch_layer_slots(const Shape &s, const LayerDev &L, const Scratch &S, const float *xn, float *out, int T,
                              int exact, int debug, hipStream_t st, int down_only = 0);
/* The shapes the integer kernels take: n_embd % 256 == 0 (the reference's fast gate,
 * src/model.c:1090-1093) and n_ff_exp % 64 == 0 (they pair 32-blocks). */
inline bool integer_grid_shape(int E, int F) { return E % 256 == 0 && F % 64 == 0; }
/* down_only: the down rows, the debug copies and the combine alone, after the integer kernels'
 * routing and gate/up (with SwiGLU) have run: n_ff_exp an odd multiple of 32, whose down rows
 * the integer kernels do not pair. */
/* Expert types the integer kernels take (the quantised types of qms_fast_supported); layers
 * with F32, F16 or Q8_0 expert tensors run slot by slot. */
inline bool integer_expert_types(int gt, int ut, int dt)
{
    auto q = [](int t) { return t == 2 || t == 3 || t == 14; };
    return q(gt) && q(ut) && q(dt);
}
hipError_t launch_synth_f32(uint64_t key, uint64_t n, float sigma, float *out, hipStream_t st);
hipError_t launch_synth_experts(uint64_t seed, uint32_t layer, uint32_t kind, int type, int64_t rows,
                                int64_t cols, int X, float sigma, uint8_t *base, hipStream_t st);
hipError_t launch_rmsnorm_rows(float *x, int T, int E, float eps, hipStream_t st);
/* LDS bytes of the rmsnorm kernel for rows of E floats (at most 160 KiB is launchable). */
inline size_t rmsnorm_lds_bytes(int E)
{
    const size_t sq = E % 512 == 0 ? (size_t)(E / 64) * 65 : (size_t)E;      /* squares, in doubles */
    return sq * 8;
}
/* y = rmsnorm(x) * w per row of E floats; with add (not NULL) x += add first, stored back.
 * walk: form every row's sum in order (else only rows the bracket leaves open); rows that do
 * are counted into *walked when it is not NULL. */
hipError_t launch_rmsnorm(float *x, const float *add, const float *w, float *y, int T, int E, float eps,
                          int walk, unsigned long long *walked, hipStream_t st);
hipError_t launch_add_rows(float *h, const float *d, size_t n, hipStream_t st);
/* dst = h + d over n floats (dst may be h). */
hipError_t launch_add_rows_to(float *dst, const float *h, const float *d, size_t n, hipStream_t st);

/* The rmsnorm of the one-token router launch (launch_route_norm): xn = rmsnorm(h + add) * w
 * (add and w may be null), stored to xn_out; h + add stored to h_out when add is not null
 * (h_out must then differ from h). */
struct NormIn {
    const float *h, *add, *w;
    float *h_out, *xn_out;
    float eps;
    int walk;
    unsigned long long *walked;
};
/* Row widths the fused launch takes. */
inline bool route_norm_fits(int E) { return E % 512 == 0 && E <= 4096; }
/* launch_route for one token with the rmsnorm in front (route_norm_kernel). */
hipError_t launch_route_norm(const Shape &s, const LayerDev &L, const Scratch &S, const NormIn &n, hipStream_t st);
hipError_t launch_set_col0(float *m, int rows, int stride, const float *vals, float fill, hipStream_t st);
hipError_t launch_silu(const float *x, int n, float *out, hipStream_t st);
hipError_t launch_exp(const double *x, int n, double *out, hipStream_t st);
hipError_t launch_copy(void *dst, const void *src, size_t bytes, hipStream_t st);
/* p[0 .. n-1] = v (a kernel, not a memset node: safe inside a captured graph). */
hipError_t launch_call_reset(const Scratch &S, hipStream_t st);
/* The dense rows kernel. Where dense_mx_takes or dense_pairs_taken the input records are formed first
 * into xqk: MFMA records (dense_record_bytes), whose flag word takes epoch (unique per call) when
 * one is outside the MFMA kernels' scaled range, or pair records. *records: xqk holds the MFMA records
 * of this call's rows (formed by an earlier launch of the call); updated. NULL: no MFMA kernels (xqk
 * smaller or NULL). */
inline size_t dense_record_bytes(size_t T, size_t C) { return 256 + T * (C / 32) * kMxRec; }
hipError_t launch_dense(const DenseArgs &a, int type, uint8_t *xqk, uint64_t epoch, bool *records, hipStream_t st);
/* matmul_exact for every matrix of a call (--exact, or an F16 / Q8_0 matrix in the call). */
hipError_t launch_dense_exact(const DenseArgs &args, int type, hipStream_t st);
/* matmul_exact rows of one stacked expert tensor for every slot (qmsg_chain.hip): slot s's input
 * is row slot_t[s] of x (by_token) or row s; y[s * y_stride + row]. With up (same rows, cols and
 * type) m is the gate tensor and y takes silu(gate) * up; gu, if not NULL, [slot][2 rows] takes
 * the gate and up rows. max_tiles bounds the slot tiles of T tokens. */
struct ChainRows {
    const uint8_t *w;
    uint64_t rb, eb;
    int type, rows, cols, by_token;
    const float *x;
    float *y;
    int y_stride;
};
/* Input rows the chain kernels stage whole in LDS: C + 4 floats a row, blocks as [g][8]. A lane
 * reads its group's words of the block after the one it multiplies, so after the last block those
 * of block C / 32, which it does not use: of the next row, or past the last row the 28 floats that
 * chain_rows_lds adds. */
__host__ __device__ constexpr int chain_row_floats(int C) { return C + 4; }
__host__ __device__ constexpr int chain_row_read(int block, int group, int quad) { return 32 * block + 8 * group + 4 * quad; }
constexpr size_t chain_rows_lds(int rows, int C) { return ((size_t)rows * (size_t)chain_row_floats(C) + 28) * 4; }
hipError_t launch_chain_rows(const char *name, const ChainRows &m, const ChainRows *up, const Scratch &S, int T,
                             int max_tiles, float *gu, hipStream_t st);
hipError_t launch_block_dots(const uint8_t *base, int type, uint64_t rb, uint64_t eb, int n, const int32_t *expert,
                             const int32_t *row, const int32_t *block, const Q8 *xq, int32_t *out,
                             hipStream_t st);

}  // namespace qmsg

#endif /* QMSG_INTERNAL_H */
