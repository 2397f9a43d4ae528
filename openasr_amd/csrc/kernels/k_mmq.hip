// k_mmq.hip -- GGML_OP_MUL_MAT on Q4_K / Q8_0 weights for wide activation
// batches (prefill, the audio prefix, N > 16) on the int8 matrix cores.
// Call site: crates/openasr-core/src/ggml_runtime/cpu_graph.rs:3652-3686.
//
// A workgroup computes a tile of 16 RW rows x 16 GRPS columns with RW KW
// waves: K group kg (RW waves of 16 rows each, all columns) takes the
// 256-element K slices kg, kg + KW, ..., so every weight fragment a wave
// loads feeds GRPS column groups. A slice's activations (quants, scales and,
// for Q4_K, the 32-element sums of the tile's columns) are staged in LDS by
// its group, double-buffered: right after a round's barrier the workgroup
// requests the next round's activations and weights into registers, computes
// the current slices from LDS, and stores the next ones into the other
// buffers at the top of the next iteration -- one barrier a round, the next
// round's loads in flight under this round's arithmetic. A buffer is written
// again only after the following barrier, which every wave reaches after its
// reads of it. The groups' sums are added through LDS at the end.
//
// What bounds it: with tiles for every CU the exact per-block epilogue on the
// VALU (64 x 64 tiles, one group); with few tiles the round trip of a slice's
// loads, K / 256 of them in turn (896 x 3584 x 78 Q8_0: 48 workgroups, 14
// slices, 42 us), which the K groups take side by side. The launch picks the
// form by the number of tiles.
//
// The arithmetic of a block unit is the GEMV's (mfma_units.h): exact block
// terms, added in f64. A group walks its slices in order and the groups are
// added in order; against one walk of K only the f64 rounding of the order
// moves (2^-53 of a partial sum), which reaches the rounded f32 result about
// once in 2^28 values.
//
// Tiles are dealt to the XCDs in contiguous runs (workgroup i runs on XCD
// i % 8): XCD x takes tiles [x P, (x + 1) P), the column blocks of a row tile
// adjacent, so a weight tile is fetched into one XCD's L2 and read there by
// all of its column blocks.
#include "../mi355x_common.h"
#include "../ops.h"
#include "../mfma_units.h"

namespace mi355x {

constexpr int kMmqRows = 64;
constexpr int kMmqCols = 64;
constexpr int kMmqPad = 16;  // bytes of padding per staged column (LDS banks)
constexpr int kMmqXcds = 8;

struct mmq_args {
    const char * W;
    int64_t row_bytes, M, K;
    const int8_t * aq;
    const float * ad;
    const int16_t * ass;
    int N;
    char * dst;
    int64_t dst_nb1;
    int64_t col_blocks, tiles, per_xcd;
    gemm_float_epi epi;  // bias, residual (laid out as dst), GELU_ERF
    // sibling products of the same activations (rows [sub_m0[i],
    // sub_m0[i + 1]) are product i: weights, contiguous output, bias)
    int nsub;
    int64_t sub_m0[kGemmFloatMaxSubs + 2];
    const char * sub_W[kGemmFloatMaxSubs + 1];
    char * sub_dst[kGemmFloatMaxSubs + 1];
    const float * sub_bias[kGemmFloatMaxSubs + 1];
    bool sub_f16[kGemmFloatMaxSubs + 1];
};

// the activations of one K slice of the tile's 16 GRPS columns
template <int GRPS>
struct mmq_slice {
    int8_t q[16 * GRPS][256 + kMmqPad];
    float d[8][16 * GRPS];     // Q4_K: [0][col] the super-block scale; Q8_0: [block][col]
    int16_t ss[16 * GRPS][8];  // Q4_K: the 32-element sums
};

// this thread's share of a slice, held in registers between its request and
// its store into LDS
template <int GRPS, int RW>
struct mmq_act {
    uint4 q[4 * GRPS / RW];
    float d[4];
    uint4 ss;
};

// t: the thread's index among the 64 RW threads that stage the slice
template <int WT, int GRPS, int RW>
__device__ __forceinline__ void mmq_act_load(const mmq_args & a, int t, int n0, int ncol, int64_t ks,
                                             mmq_act<GRPS, RW> & r) {
    static_assert(GRPS <= 2 * RW, "a thread stages at most four scales");
#pragma unroll
    for (int u = 0; u < 4 * GRPS / RW; u++) {
        const int idx = t + 64 * RW * u, col = idx >> 4, piece = idx & 15;
        const int64_t kk = ks * 256 + piece * 16;
        const bool ok = col < ncol && kk < a.K;
        // clamped address, unconditional load: masked when stored
        r.q[u] = *(const uint4 *) (a.aq + (int64_t) (n0 + (ok ? col : 0)) * a.K + (ok ? kk : 0));
    }
    if constexpr (WT == GGML_TYPE_Q4_K) {
        const int64_t nsb = a.K / 256;
        const int col = t < ncol ? t : 0;
        if (t < 16 * GRPS) {
            r.d[0] = a.ad[(int64_t) (n0 + col) * nsb + ks];
            r.ss = *(const uint4 *) (a.ass + ((int64_t) (n0 + col) * nsb + ks) * 8);
        }
    } else {
        const int64_t nblk = a.K / 32;
        const int col = (t >> 1) < ncol ? (t >> 1) : 0, h = t & 1;
        if (t < 32 * GRPS) {
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int64_t b = ks * 8 + 4 * h + j;
                r.d[j] = a.ad[(int64_t) (n0 + col) * nblk + (b < nblk ? b : nblk - 1)];
            }
        }
    }
}

template <int WT, int GRPS, int RW>
__device__ __forceinline__ void mmq_act_store(const mmq_args & a, int t, int ncol, int64_t ks,
                                              const mmq_act<GRPS, RW> & r, mmq_slice<GRPS> & S) {
#pragma unroll
    for (int u = 0; u < 4 * GRPS / RW; u++) {
        const int idx = t + 64 * RW * u, col = idx >> 4, piece = idx & 15;
        const bool ok = col < ncol && ks * 256 + piece * 16 < a.K;
        *(uint4 *) &S.q[col][piece * 16] = ok ? r.q[u] : make_uint4(0, 0, 0, 0);
    }
    if constexpr (WT == GGML_TYPE_Q4_K) {
        if (t < 16 * GRPS) {
            const bool ok = t < ncol;
            S.d[0][t] = ok ? r.d[0] : 0.0f;
            *(uint4 *) &S.ss[t][0] = ok ? r.ss : make_uint4(0, 0, 0, 0);
        }
    } else {
        const int64_t nblk = a.K / 32;
        if (t < 32 * GRPS) {
            const int col = t >> 1, h = t & 1;
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const bool ok = col < ncol && ks * 8 + 4 * h + j < nblk;
                S.d[4 * h + j][col] = ok ? r.d[j] : 0.0f;
            }
        }
    }
}

// this lane's weights of one slice: Q4_K one super-block of its row, Q8_0
// eight blocks (past the end of K: the row's last block, never used)
struct mmq_w4 {
    uint4 hdr;
    long q[4];
};
struct mmq_w8 {
    long q[kQ8Group];
    uint16_t ds[kQ8Group];
};

__device__ __forceinline__ void mmq_w_load(const mmq_args & a, const char * wrow, int64_t ks, int g, mmq_w4 & w) {
    (void) a;
    const char * blk = wrow + ks * 144;
    w.hdr = *(const uint4 *) blk;
#pragma unroll
    for (int c = 0; c < 4; c++) w.q[c] = *(const long *) (blk + 16 + 32 * c + 8 * g);
}

__device__ __forceinline__ void mmq_w_load(const mmq_args & a, const char * wrow, int64_t ks, int g, mmq_w8 & w) {
    const int64_t nblk = a.K / 32;
    const uint16_t * wsc = (const uint16_t *) (wrow + a.K);
#pragma unroll
    for (int bb = 0; bb < kQ8Group; bb++) {
        const int64_t b = ks * 8 + bb < nblk ? ks * 8 + bb : nblk - 1;
        w.q[bb] = *(const long *) (wrow + b * 32 + 8 * g);
        w.ds[bb] = wsc[b];
    }
}

template <int GRPS>
__device__ __forceinline__ void mmq_compute(const mmq_args & a, const mmq_slice<GRPS> & S, const mmq_w4 & w, int64_t ks,
                                            int r, int g, double (&acc)[GRPS][4]) {
    (void) a;
    (void) ks;
#pragma unroll
    for (int grp = 0; grp < GRPS; grp++) {
        const int8_t * acol = &S.q[grp * 16 + r][0];
        long af[8];
#pragma unroll
        for (int j = 0; j < 8; j++) af[j] = *(const long *) (acol + 32 * j + 8 * g);
        const float4 d4 = *(const float4 *) &S.d[0][grp * 16 + 4 * g];
        const float ad[4] = {d4.x, d4.y, d4.z, d4.w};
        float ssa[2];
        q4k_ssum_operand(&S.ss[grp * 16 + r][0], true, g, ssa);  // columns past N were staged as zeros
        q4k_unit(w.hdr, w.q, af, ad, ssa, acc[grp]);
    }
}

template <int GRPS>
__device__ __forceinline__ void mmq_compute(const mmq_args & a, const mmq_slice<GRPS> & S, const mmq_w8 & w, int64_t ks,
                                            int r, int g, double (&acc)[GRPS][4]) {
    const int64_t nblk = a.K / 32;
    const int nb = (int) (nblk - ks * 8 < kQ8Group ? nblk - ks * 8 : kQ8Group);
    // block by block (each (row, column) sum still takes its blocks in order),
    // the column groups inner: a block's weights and scale serve four groups
#pragma unroll
    for (int u = 0; u < kQ8Group; u++) {
        if (u >= nb) break;
#pragma unroll
        for (int grp = 0; grp < GRPS; grp++) {
            const long af = *(const long *) (&S.q[grp * 16 + r][32 * u + 8 * g]);
            const float4 d4 = *(const float4 *) &S.d[u][grp * 16 + 4 * g];
            const float da[4] = {d4.x, d4.y, d4.z, d4.w};
            q8_0_block(af, w.q[u], w.ds[u], da, acc[grp]);
        }
    }
}

// sibling products: row_tile's product becomes the launch's (a's weights, rows
// and output), row_tile its tile; selected with constant indices (an index
// into the argument arrays would put them in scratch memory)
template <bool HALF>
__device__ __forceinline__ void mmq_pick_product(mmq_args & a, int64_t & row_tile, int tile_rows) {
    static_assert(kGemmFloatMaxSubs == 2, "product selection below");
    if (a.nsub <= 0) return;
    const int64_t r0 = row_tile * tile_rows;
    int64_t base = 0, mend = a.sub_m0[1];
    const char * sw = a.sub_W[0];
    char * sd = a.sub_dst[0];
    const float * sb = a.sub_bias[0];
    bool sh = HALF && a.sub_f16[0];
    if (r0 >= a.sub_m0[1]) {
        base = a.sub_m0[1], mend = a.sub_m0[2];
        sw = a.sub_W[1], sd = a.sub_dst[1], sb = a.sub_bias[1], sh = HALF && a.sub_f16[1];
    }
    if (a.nsub >= 2 && r0 >= a.sub_m0[2]) {
        base = a.sub_m0[2], mend = a.sub_m0[3];
        sw = a.sub_W[2], sd = a.sub_dst[2], sb = a.sub_bias[2], sh = HALF && a.sub_f16[2];
    }
    row_tile -= base / tile_rows;
    a.M = mend - base;
    a.W = sw;
    a.dst = sd;
    a.dst_nb1 = a.M * (sh ? 2 : 4);  // each product's output is contiguous
    a.epi.bias = sb;
    a.epi.f16_out = sh;
}

// HALF: some product's result is f16 (a branch in every store otherwise, 1-2 %)
template <int WT, int GRPS, int RW, int KW, bool HALF>
__global__ __launch_bounds__(64 * RW * KW) void k_mmq(mmq_args a) {
    constexpr int kRows = 16 * RW;
    __shared__ __align__(16) mmq_slice<GRPS> s_buf[2][KW];
    using wregs = typename std::conditional<WT == GGML_TYPE_Q4_K, mmq_w4, mmq_w8>::type;
    // contiguous runs of tiles per XCD
    const int64_t id = blockIdx.x;
    const int64_t t = (id % kMmqXcds) * a.per_xcd + id / kMmqXcds;
    if (t >= a.tiles) return;  // before any barrier: the whole workgroup leaves
    int64_t row_tile = t / a.col_blocks;
    const int64_t col_block = t % a.col_blocks;
    mmq_pick_product<HALF>(a, row_tile, kRows);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int rw = KW > 1 ? wave % RW : wave, kg = KW > 1 ? wave / RW : 0;
    const int st = KW > 1 ? (int) threadIdx.x % (64 * RW) : (int) threadIdx.x;
    const int r = lane & 15, g = lane >> 4;
    const int64_t row = row_tile * kRows + rw * 16 + r;
    const bool row_ok = row_tile * kRows + rw * 16 < a.M;  // uniform per wave
    const int n0 = (int) (col_block * 16 * GRPS);
    const int ncol = min(16 * GRPS, a.N - n0);
    const int64_t nks = (a.K + 255) / 256;
    const char * wrow = a.W + (row_ok ? row : 0) * a.row_bytes;
    double acc[GRPS][4];
#pragma unroll
    for (int grp = 0; grp < GRPS; grp++)
#pragma unroll
        for (int i = 0; i < 4; i++) acc[grp][i] = 0.0;
    mmq_act<GRPS, RW> act;
    wregs wn;
    if constexpr (KW == 1) {
        // one group: a loop of its own, as the groups' guards cost it 2-6 %
        mmq_act_load<WT, GRPS, RW>(a, st, n0, ncol, 0, act);
        mmq_w_load(a, wrow, 0, g, wn);
        for (int64_t ks = 0; ks < nks; ks++) {
            mmq_slice<GRPS> & S = s_buf[ks & 1][0];
            mmq_act_store<WT, GRPS, RW>(a, st, ncol, ks, act, S);
            const wregs w = wn;
            __syncthreads();
            if (ks + 1 < nks) {
                mmq_act_load<WT, GRPS, RW>(a, st, n0, ncol, ks + 1, act);
                mmq_w_load(a, wrow, ks + 1, g, wn);
            }
            if (row_ok) mmq_compute<GRPS>(a, S, w, ks, r, g, acc);
        }
    } else {
        // K group kg takes the slices kg, kg + KW, ...: every group runs the
        // same number of rounds (barriers), the groups past the last slice idle
        if (kg < nks) {
            mmq_act_load<WT, GRPS, RW>(a, st, n0, ncol, kg, act);
            mmq_w_load(a, wrow, kg, g, wn);
        }
        int buf = 0;
        for (int64_t k0 = 0; k0 < nks; k0 += KW, buf ^= 1) {
            const int64_t ks = k0 + kg;
            mmq_slice<GRPS> & S = s_buf[buf][kg];
            if (ks < nks) mmq_act_store<WT, GRPS, RW>(a, st, ncol, ks, act, S);
            const wregs w = wn;
            __syncthreads();
            if (ks + KW < nks) {
                mmq_act_load<WT, GRPS, RW>(a, st, n0, ncol, ks + KW, act);
                mmq_w_load(a, wrow, ks + KW, g, wn);
            }
            if (row_ok && ks < nks) mmq_compute<GRPS>(a, S, w, ks, r, g, acc);
        }
        // the groups' sums through the staging buffers, added in group order
        double * s_acc = (double *) &s_buf[0][0];
        static_assert(sizeof(s_buf) >= sizeof(double) * 256 * GRPS * RW * (KW - 1), "the staging buffers hold the sums");
        __syncthreads();  // the last slices are read
        if (kg > 0) {
#pragma unroll
            for (int grp = 0; grp < GRPS; grp++)
#pragma unroll
                for (int i = 0; i < 4; i++)
                    s_acc[(((kg - 1) * RW + rw) * 4 * GRPS + 4 * grp + i) * 64 + lane] = acc[grp][i];
        }
        __syncthreads();
        if (kg > 0) return;
#pragma unroll
        for (int k = 0; k < KW - 1; k++)
#pragma unroll
            for (int grp = 0; grp < GRPS; grp++)
#pragma unroll
                for (int i = 0; i < 4; i++) acc[grp][i] += s_acc[((k * RW + rw) * 4 * GRPS + 4 * grp + i) * 64 + lane];
    }
    if (!row_ok) return;
    // the adds, then (GELU_ERF) the lane's GELUs together, then the stores
    float o[4 * GRPS];
#pragma unroll
    for (int grp = 0; grp < GRPS; grp++) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int n = n0 + grp * 16 + 4 * g + i;
            float v = (float) acc[grp][i];
            if (n < a.N) {
                if (a.epi.bias) v = v + a.epi.bias[row];
                if (a.epi.res) v = v + a.epi.res[(int64_t) n * a.M + row];
            }
            o[grp * 4 + i] = v;
        }
    }
    if (a.epi.gelu_erf) gelu_erf_det_n<4 * GRPS>(o);
#pragma unroll
    for (int grp = 0; grp < GRPS; grp++) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int n = n0 + grp * 16 + 4 * g + i;
            if (n >= a.N) continue;
            if (HALF && a.epi.f16_out) *(uint16_t *) (a.dst + (int64_t) n * a.dst_nb1 + row * 2) = float_to_half_bits(o[grp * 4 + i]);
            else *(float *) (a.dst + (int64_t) n * a.dst_nb1 + row * 4) = o[grp * 4 + i];
        }
    }
}

template <int V>
using mmq_int = std::integral_constant<int, V>;

bool mmq_supported(int wtype, int64_t M, int64_t K) {
    if (M % 16 != 0) return false;
    if (wtype == GGML_TYPE_Q4_K) return K % 256 == 0;
    if (wtype == GGML_TYPE_Q8_0) return K % 32 == 0;
    return false;
}

void launch_mmq(int wtype, const char * W, int64_t row_bytes, int64_t M, int64_t K, const act_buffers & act,
                int64_t N, char * dst, int64_t dst_nb1, hipStream_t stream, int n_cu, const gemm_float_epi & epi,
                const gemm_float_sub * subs, int nsub) {
    mmq_args a;
    a.nsub = 0;
    int64_t m_all = M;
    if (nsub > 0 && nsub <= kGemmFloatMaxSubs && M % kMmqRows == 0 && !epi.res && !epi.gelu_erf) {
        a.nsub = nsub;
        a.sub_m0[0] = 0;
        a.sub_W[0] = W;
        a.sub_dst[0] = dst;
        a.sub_bias[0] = epi.bias;
        a.sub_f16[0] = epi.f16_out;
        for (int i = 0; i < nsub; i++) {
            a.sub_m0[i + 1] = m_all;
            a.sub_W[i + 1] = subs[i].a;
            a.sub_dst[i + 1] = subs[i].d;
            a.sub_bias[i + 1] = subs[i].bias;
            a.sub_f16[i + 1] = subs[i].f16_out;
            m_all += subs[i].M;
        }
        a.sub_m0[nsub + 1] = m_all;
    } else if (nsub > 0) {
        // not joinable: each product on its own
        launch_mmq(wtype, W, row_bytes, M, K, act, N, dst, dst_nb1, stream, n_cu, epi);
        for (int i = 0; i < nsub; i++) {
            gemm_float_epi ei;
            ei.bias = subs[i].bias;
            ei.f16_out = subs[i].f16_out;
            launch_mmq(wtype, subs[i].a, row_bytes, subs[i].M, K, act, N, subs[i].d, subs[i].M * (ei.f16_out ? 2 : 4),
                       stream, n_cu, ei);
        }
        return;
    }
    a.epi = epi;
    a.W = W;
    a.row_bytes = row_bytes;
    a.M = M;
    a.K = K;
    a.aq = act.q;
    a.ad = act.d;
    a.ass = act.ssum;
    a.N = (int) N;
    a.dst = dst;
    a.dst_nb1 = dst_nb1;
    bool half = epi.f16_out;
    for (int i = 0; i < nsub; i++) half = half || subs[i].f16_out;
    auto form = [&](auto grps, auto rw, auto kw) {
        constexpr int G = decltype(grps)::value, R = decltype(rw)::value, KW = decltype(kw)::value;
        a.col_blocks = (N + 16 * G - 1) / (16 * G);
        a.tiles = (m_all + 16 * R - 1) / (16 * R) * a.col_blocks;
        a.per_xcd = (a.tiles + kMmqXcds - 1) / kMmqXcds;
        auto go = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, dim3((unsigned) (a.per_xcd * kMmqXcds)), dim3(64 * R * KW), 0, stream, a);
        };
        if (wtype == GGML_TYPE_Q4_K && half) go(k_mmq<GGML_TYPE_Q4_K, G, R, KW, true>);
        else if (wtype == GGML_TYPE_Q4_K) go(k_mmq<GGML_TYPE_Q4_K, G, R, KW, false>);
        else if (half) go(k_mmq<GGML_TYPE_Q8_0, G, R, KW, true>);
        else go(k_mmq<GGML_TYPE_Q8_0, G, R, KW, false>);
    };
    // The form by how many 64 x 64 tiles there are for the CUs: fewer tiles,
    // more and smaller workgroups and more K groups in flight. Per call with
    // the activation quantization and the wait, us, Q8_0 / Q4_K at 256 CUs
    // (left: the form before, 64 x 32 tiles of one K group below 256 tiles):
    //   28 tiles  896 x 3584 x 78    50.1 -> 28.0 / 32.2 -> 23.3 (16-row form; 32-row 31.8 / 24.3)
    //   32 tiles  1024 x 3072 x 119  45.3 -> 25.9 / 30.2 -> 22.3
    //   64 tiles  2048 x 6144 x 100  77.2 -> 48.5 / 46.8 -> 32.2 (32-row form, 4 groups; 16-row 51.2 / 33.1)
    //   98 tiles  896 x 3584 x 390   52.1 -> 46.1 / 35.4 -> 32.8 (2 groups; 4 groups 49.8 / 35.7)
    //   192 tiles 6144 x 2048 x 100  52.5 -> 45.9 / 31.0 -> 29.6
    //   256 tiles 1024 x 2048 x 1000 49.6 -> 45.8 / 37.5 -> 35.7 (64 x 64 tiles, 2 groups)
    //   392 tiles 3584 x 896 x 390   36.7 with one group, 39.0 with two
    const int64_t tiles = (m_all + kMmqRows - 1) / kMmqRows * ((N + kMmqCols - 1) / kMmqCols);
    const bool deep = K > 512;  // slices for four K groups (K = 384: two)
    if (deep && 6 * tiles <= n_cu) form(mmq_int<2>{}, mmq_int<1>{}, mmq_int<4>{});
    else if (deep && 4 * tiles <= n_cu) form(mmq_int<2>{}, mmq_int<2>{}, mmq_int<4>{});
    else if (4 * tiles <= 3 * n_cu) form(mmq_int<2>{}, mmq_int<2>{}, mmq_int<2>{});
    else if (tiles <= n_cu) form(mmq_int<4>{}, mmq_int<4>{}, mmq_int<2>{});
    else form(mmq_int<4>{}, mmq_int<4>{}, mmq_int<1>{});
}

}  // namespace mi355x
