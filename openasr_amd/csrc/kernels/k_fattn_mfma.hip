// k_fattn_mfma.hip -- GGML_OP_FLASH_ATTN_EXT with more than one query
// position (prefill chunks, the audio encoders' self attention) at the
// default precision, on the matrix cores. Call site of the op:
// crates/openasr-core/src/ggml_runtime/cpu_graph.rs:4144-4215; the precision
// contract: Default is the backend's fastest validated implementation, F32
// ggml's full-precision contract (cpu_graph.rs:129-133, set per graph,
// models/qwen/llm_transformer.rs:3044-3053). F32 graphs and single-query
// (decode) steps keep the exact chunked form of k_fattn.hip.
//
// Arithmetic (float tolerance, the ggml GPU backends' flash attention): the
// query rows rounded to f16, S^T = K Q^T on v_mfma_f32_16x16x32_f16 (f16
// products, f32 sums), S * scale * log2(e) + mask * log2(e) in f32, an
// online softmax over 64-position tiles in f32 with exp2 (running max m, sum
// l, the output rescaled by 2^(m_old - m_new)), P rounded to f16 for
// O^T = V^T P^T on the same MFMA, out = O / l (0 for a row with no open
// position).
//
// Work: a workgroup of four waves owns 64 rows -- 64 / g queries times the
// g query heads of one kv head of one sequence -- so each K/V tile is read
// once for g heads; wave w owns rows 16 w .. 16 w + 15. MFMA operand layouts
// (16x16x32): A lane l = row l % 16, k 8 (l / 16) .. + 7; B lane l = k
// 8 (l / 16) .. + 7, column l % 16; result lane l = rows 4 (l / 16) .. + 3,
// column l % 16. The scores are computed transposed (rows = positions,
// columns = the wave's rows), so a lane holds 16 positions of one row: the
// softmax is lane-local but for two cross-lane steps, and its P values are
// the lane's own B operand of the P V product (the k slots ordered to match,
// V^T read in that order) -- P never goes through LDS. Per 64-position tile:
// K rows staged in LDS (rows padded against bank conflicts), V staged
// transposed ([dim][position]), the mask as f32.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "../mi355x_common.h"
#include "../ops.h"

namespace mi355x {

namespace {

constexpr int kFmRows = 64;       // rows a workgroup owns
constexpr int kFmTile = 64;       // KV positions a tile
constexpr int kFmThreads = 256;
constexpr int kFmMaxSpan = 8192;  // positions one split covers (its live bits sit in LDS)
constexpr uint16_t kFmNegInf = 0xFC00u;

typedef _Float16 fm_h8 __attribute__((ext_vector_type(8)));
typedef float fm_f4 __attribute__((ext_vector_type(4)));
typedef uint32_t fm_u4 __attribute__((ext_vector_type(4)));  // 16 bytes (a native vector: copies stay in registers)

__device__ __forceinline__ fm_h8 fm_load8(const _Float16 * p) { return *(const fm_h8 *) p; }

// Mask entries pos .. pos + 7 of one mask row (f16 bits), in two steps so
// that a thread's loads issue back to back and are waited for only where the
// values are used. fm_mask_load: unconditional loads. MM (the mask form, one
// per kernel): 0 no mask (zeros); 1 16-byte rows -- the aligned 16-byte
// piece at pos, or the last piece holding an entry below n_kv when pos is
// past it (an aligned 16-byte piece holding a valid entry lies in that
// entry's page); 3 4-byte rows -- four word loads the same way; 2 other
// rows -- eight 2-byte loads, indexes clamped below n_kv. fm_mask_fix:
// positions at or past n_kv become -inf.
template <int MM>
__device__ __forceinline__ fm_u4 fm_mask_load(const uint16_t * row, int pos, int n_kv) {
    if constexpr (MM == 0) {
        return fm_u4{0, 0, 0, 0};
    } else if constexpr (MM == 1) {
        return *(const fm_u4 *) (row + min(pos, (n_kv - 1) & ~7));
    } else if constexpr (MM == 3) {
        // 4-byte rows: four word loads, clamped to the last word holding an
        // entry below n_kv (pos is even; a word holding a valid entry lies in
        // that entry's page)
        const uint32_t * w = (const uint32_t *) row;
        const int wi = pos >> 1, wl = (n_kv - 1) >> 1;
        return fm_u4{w[min(wi, wl)], w[min(wi + 1, wl)], w[min(wi + 2, wl)], w[min(wi + 3, wl)]};
    } else {
        uint32_t h[8];
#pragma unroll
        for (int j = 0; j < 8; j++) h[j] = row[min(pos + j, n_kv - 1)];
        return fm_u4{h[0] | (h[1] << 16), h[2] | (h[3] << 16), h[4] | (h[5] << 16), h[6] | (h[7] << 16)};
    }
}

__device__ __forceinline__ fm_u4 fm_mask_fix(fm_u4 m, int pos, int n_kv) {
    if (pos + 8 <= n_kv) return m;
    uint32_t w[4] = {m.x, m.y, m.z, m.w};
#pragma unroll
    for (int j = 0; j < 4; j++) {
        if (pos + 2 * j >= n_kv) w[j] = (w[j] & 0xFFFF0000u) | kFmNegInf;
        if (pos + 2 * j + 1 >= n_kv) w[j] = (w[j] & 0xFFFFu) | ((uint32_t) kFmNegInf << 16);
    }
    return fm_u4{w[0], w[1], w[2], w[3]};
}

// bit j set when entry j of the eight is not -inf
__device__ __forceinline__ uint32_t fm_open_bits(fm_u4 m) {
    const uint32_t w[4] = {m.x, m.y, m.z, m.w};
    uint32_t bits = 0;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        bits |= ((w[j] & 0xFFFFu) != kFmNegInf ? 1u : 0u) << (2 * j);
        bits |= ((w[j] >> 16) != kFmNegInf ? 1u : 0u) << (2 * j + 1);
    }
    return bits;
}

// one more split (maximum m in base-2 exponent units, sum l) into the merged
// state (M, L): the factors wa of the merged output and wb of the split's. A
// split with nothing open changes nothing; merging into nothing is exact.
__device__ __forceinline__ void fm_merge(float & M, float & L, float m, float l, float & wa, float & wb) {
    const float mn = fmaxf(M, m);
    wa = M == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(M - mn);
    wb = m == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m - mn);
    L = L * wa + l * wb;
    M = mn;
}

}  // namespace

// Per workgroup: (1) the mask of its queries over its split of the span is
// scanned once into per-position "seen by some query" bits in LDS; tiles with
// none are skipped and V rows no query sees are staged as zeros (0 x V stays
// 0 whatever the cache holds there). (2) Live tiles are software-pipelined:
// the next live tile's K / V / mask are loaded into registers while the
// current one is on the matrix cores.
//
// KV32: K and V are f32 (the encoders' head views of their projections),
// staged rounded to f16 -- what a copy to f16 tensors ahead of the launch
// would hold: that launch (6.6 us a layer of a 30 s encode) goes, the
// attention itself takes 21 us (23 over f16 copies, before its unmasked tiles).
// Reading an f32 mask here as well, in place of its 5 us cast, measured 27.5 us:
// its rows on 4 bytes take a load an entry.
//
// MG: the workgroup takes every split of its rows in turn and merges
// their states in registers (fm_merge, in split order, what the combine
// launch computes), writing no partials.
template <int D, int MM, bool MG, bool KV32>
__global__ __launch_bounds__(kFmThreads) void k_fattn_mfma(fattn_args a, float * __restrict__ out,
                                                           float * __restrict__ part) {
    constexpr int KS = D / 32;  // k steps of the score MFMA
    constexpr int NT = D / 16;  // output column tiles
    constexpr int KP = D + 8;   // padded K row (halves)
    constexpr int VP = kFmTile + 8;
    constexpr int PC = D / 8;                                   // 16-byte pieces of a K / V row
    constexpr int KLD = kFmTile * PC / kFmThreads;              // K pieces a thread stages
    constexpr int VLD = (kFmTile / 2) * PC / kFmThreads;        // V piece pairs (two positions) a thread stages
    constexpr int MLD = kFmRows * (kFmTile / 8) / kFmThreads;   // 8-entry mask pieces a thread stages (at most)
    static_assert(KLD >= 1 && VLD >= 1 && MLD >= 1, "staging split");
    __shared__ __align__(16) _Float16 s_k[kFmTile][KP];
    __shared__ __align__(16) _Float16 s_vt[D][VP];
    __shared__ __align__(16) float s_m[kFmRows][kFmTile + 4];  // mask x log2(e), -inf kept
    __shared__ uint32_t s_open[kFmMaxSpan / 32];
    __shared__ uint32_t s_masked[kFmMaxSpan / kFmTile];  // tile: some mask entry is not zero
    const int tid = (int) threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int g = a.hq / a.hkv, qpw = kFmRows / g;  // queries a workgroup
    // Workgroup b is dispatched to XCD b % 8: each XCD gets a contiguous run
    // of (query block, kv head / sequence, split) coordinates, query blocks
    // fastest, so the query blocks reading the same K / V tiles share an L2.
    const int q_blocks = (a.n_q + qpw - 1) / qpw, n_blk = (int) gridDim.x;
    int b = (int) blockIdx.x;
    if (n_blk % 8 == 0) b = (b % 8) * (n_blk / 8) + b / 8;
    const int qb = b % q_blocks, hs = (b / q_blocks) % (a.hkv * a.n_seq), z = b / (q_blocks * a.hkv * a.n_seq);
    const int kvh = hs % a.hkv, seq = hs / a.hkv;
    const int q0 = qb * qpw;
    const int nq_live = min(qpw, a.n_q - q0);
    const int kv_seq = seq / a.rk3;
    const int l16 = lane & 15, lg = lane >> 4;
    const char * kbase = a.k + (int64_t) kvh * a.k_nb2 + (int64_t) kv_seq * a.k_nb3;
    const char * vbase = a.v + (int64_t) kvh * a.v_nb2 + (int64_t) kv_seq * a.v_nb3;
    const char * mbase = MM ? a.mask + (int64_t) (seq % a.m_ne3) * a.m_nb3 : nullptr;
    auto mask_row = [&](int ql) { return (const uint16_t *) (mbase + (int64_t) (q0 + ql) * a.m_nb1); };
    // this workgroup's share of the span: tiles [t_begin, t_end) of split z
    const int n_tiles = (a.n_kv + kFmTile - 1) / kFmTile;
    const int per = (n_tiles + a.mfma_split - 1) / a.mfma_split;
    const int t_begin = MG ? 0 : z * per, t_end = MG ? n_tiles : min(n_tiles, t_begin + per);
    int z_end = t_begin + per;  // MG: the current split's last tile + 1
    const int span0 = t_begin * kFmTile;

    // registers for one tile in flight
    constexpr int EW = KV32 ? 2 : 1;  // 16-byte loads an 8-element piece takes
    fm_u4 kr[KLD][EW], vr[VLD][2][EW], mr[MLD];
    // eight elements as f16
    auto half8 = [](const fm_u4 (&r)[EW]) {
        if constexpr (!KV32) {
            return r[0];
        } else {
            fm_u4 h;
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const fm_u4 w = r[j >> 1];
                h[j] = (uint32_t) float_to_half_bits(__uint_as_float(w[2 * (j & 1)])) |
                       ((uint32_t) float_to_half_bits(__uint_as_float(w[2 * (j & 1) + 1])) << 16);
            }
            return h;
        }
    };
    auto issue = [&](int tile, bool masked) {
        const int p0 = tile * kFmTile;
        // every load unconditional (rows clamped into the span, the result
        // selected after), so they issue back to back
#pragma unroll
        for (int i = 0; i < KLD; i++) {
            const int e = tid + i * kFmThreads, p = e / PC, piece = e % PC;
#pragma unroll
            for (int w = 0; w < EW; w++)
                kr[i][w] = *(const fm_u4 *) (kbase + (int64_t) min(p0 + p, a.n_kv - 1) * a.k_nb1 + 16 * (EW * piece + w));
        }
#pragma unroll
        for (int i = 0; i < VLD; i++) {
            const int e = tid + i * kFmThreads, pair = e % (kFmTile / 2), piece = e / (kFmTile / 2);
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const int p = p0 + 2 * pair + h;
#pragma unroll
                for (int w = 0; w < EW; w++)
                    vr[i][h][w] = *(const fm_u4 *) (vbase + (int64_t) min(p, a.n_kv - 1) * a.v_nb1 + 16 * (EW * piece + w));
            }
        }
        if (!masked) return;
#pragma unroll
        for (int i = 0; i < MLD; i++) {
            const int e = tid + i * kFmThreads, ql = e >> 3, c = e & 7;
            mr[i] = fm_mask_load<MM>(mask_row(min(ql, nq_live - 1)), p0 + 8 * c, a.n_kv);
        }
        // positions past the span: their K rows (copies of the last) meet a
        // -inf mask, their V rows are not open (staged as zeros)
    };
    // the split's first tile goes out with the query rows and the mask scan
    // (one memory round trip for all three)
    issue(t_begin, true);

    // this lane's query row (the score MFMA's A operand): row 16 wave + l16,
    // dims 8 lg .. + 7 of each 32-dim step, f16-rounded
    const int q_row = 16 * wave + l16;
    const bool q_live = q0 + q_row / g < a.n_q;
    float qv[KS][8];
    {
        const float * qp = (const float *) (a.q + (int64_t) (q_live ? q0 + q_row / g : 0) * a.q_nb1 +
                                            (int64_t) (kvh * g + q_row % g) * a.q_nb2 + (int64_t) seq * a.q_nb3);
#pragma unroll
        for (int kk = 0; kk < KS; kk++) {
#pragma unroll
            for (int j = 0; j < 8; j++) qv[kk][j] = qp[32 * kk + 8 * lg + j];  // a row of query 0 for a dead row
        }
    }

    // (1) positions of the split some query of the workgroup sees
    const int words = (t_end - t_begin) * (kFmTile / 32);
    for (int w = tid; w < words; w += kFmThreads) s_open[w] = 0;
    // (the unmasked form takes the maximum before the scale: a scale above 0)
    const uint32_t all_masked = a.scale > 0.0f ? 0u : 1u;
    for (int w = tid; w < t_end - t_begin; w += kFmThreads) s_masked[w] = all_masked;
    __syncthreads();
    {
        const int pieces = (t_end - t_begin) * (kFmTile / 8);  // 8-position pieces of a row
        const int total = nq_live * pieces;
        for (int e0 = tid; e0 < total; e0 += 4 * kFmThreads) {
            fm_u4 raw[4];
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const int e = min(e0 + u * kFmThreads, total - 1);
                raw[u] = fm_mask_load<MM>(mask_row(e / pieces), span0 + 8 * (e % pieces), a.n_kv);
            }
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const int e = e0 + u * kFmThreads, c = e % pieces;
                if (e >= total) continue;
                const fm_u4 m8 = fm_mask_fix(raw[u], span0 + 8 * c, a.n_kv);
                const uint32_t bits = fm_open_bits(m8);
                if (bits) atomicOr(&s_open[c >> 2], bits << (8 * (c & 3)));
                if ((m8.x | m8.y | m8.z | m8.w) & 0x7FFF7FFFu) s_masked[c >> 3] = 1;  // -0 adds as 0
            }
        }
    }
    __syncthreads();
    auto tile_open = [&](int t) {
        const int w = (t - t_begin) * (kFmTile / 32);
        return (s_open[w] | s_open[w + 1]) != 0;
    };
    auto tile_masked = [&](int t) { return s_masked[t - t_begin] != 0; };
    auto next_open = [&](int t) {
        while (t < t_end && !tile_open(t)) t++;
        return t;
    };

    // scores are taken to base-2 exponent units in f32 (exp2 on the softmax
    // side): s = S * scale * log2(e) + mask * log2(e)
    const float qscale = a.scale * 1.4426950408889634f;
    fm_h8 qa[KS];
#pragma unroll
    for (int kk = 0; kk < KS; kk++) {
#pragma unroll
        for (int j = 0; j < 8; j++) qa[kk][j] = q_live ? (_Float16) qv[kk][j] : (_Float16) 0.0f;
    }
    // this lane's row (query / head pair): 16 wave + l16; its running max,
    // sum and O^T columns (dims 16 ct + 4 lg + i)
    float m = -INFINITY, l = 0.0f;
    fm_f4 o[NT];
    // MG: the finished splits' merged state
    float M = -INFINITY, L = 0.0f;
    fm_f4 O[NT];
#pragma unroll
    for (int ct = 0; ct < NT; ct++) {
        o[ct] = fm_f4{0.f, 0.f, 0.f, 0.f};
        if constexpr (MG) O[ct] = o[ct];
    }

    // (2) the pipeline over the open tiles
    auto stage = [&](int tile, bool masked) {
        const int rel = tile * kFmTile - span0;
#pragma unroll
        for (int i = 0; i < KLD; i++) {
            const int e = tid + i * kFmThreads, p = e / PC, piece = e % PC;
            *(fm_u4 *) &s_k[p][8 * piece] = half8(kr[i]);
        }
#pragma unroll
        for (int i = 0; i < VLD; i++) {
            const int e = tid + i * kFmThreads, pair = e % (kFmTile / 2), piece = e / (kFmTile / 2);
            fm_u4 v0 = half8(vr[i][0]), v1 = half8(vr[i][1]);
            if (masked) {  // an unmasked tile is open throughout
                const int pr = rel + 2 * pair;  // even: both positions in one word
                const uint32_t open = s_open[pr >> 5] >> (pr & 31);
                if (!(open & 1u)) v0 = fm_u4{0, 0, 0, 0};
                if (!(open & 2u)) v1 = fm_u4{0, 0, 0, 0};
            }
#pragma unroll
            for (int j = 0; j < 4; j++) {
                *(uint32_t *) &s_vt[8 * piece + 2 * j][2 * pair] = __builtin_amdgcn_perm(v1[j], v0[j], 0x05040100u);
                *(uint32_t *) &s_vt[8 * piece + 2 * j + 1][2 * pair] = __builtin_amdgcn_perm(v1[j], v0[j], 0x07060302u);
            }
        }
        if (!masked) return;
#pragma unroll
        for (int i = 0; i < MLD; i++) {
            const int e = tid + i * kFmThreads, ql = e >> 3, c = e & 7;
            if (ql >= qpw) continue;
            const fm_u4 mh = ql < nq_live ? fm_mask_fix(mr[i], tile * kFmTile + 8 * c, a.n_kv)
                                          : fm_u4{0xFC00FC00u, 0xFC00FC00u, 0xFC00FC00u, 0xFC00FC00u};
            fm_f4 lo, hi;
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const uint32_t w = mh[j];
                const float e0 = half_bits_to_float((uint16_t) (w & 0xFFFFu)), e1 = half_bits_to_float((uint16_t) (w >> 16));
                const float f0 = e0 * 1.4426950408889634f, f1 = e1 * 1.4426950408889634f;
                if (j < 2) {
                    lo[2 * j] = f0;
                    lo[2 * j + 1] = f1;
                } else {
                    hi[2 * j - 4] = f0;
                    hi[2 * j - 3] = f1;
                }
            }
            *(fm_f4 *) &s_m[ql][8 * c] = lo;
            *(fm_f4 *) &s_m[ql][8 * c + 4] = hi;
        }
    };

    int tile = next_open(t_begin);
    bool masked = tile < t_end && tile_masked(tile);
    if (tile < t_end && tile != t_begin) issue(tile, masked);  // the first tile was not open
    if constexpr (MG) {
        while (z_end <= tile) z_end += per;
    }
    while (tile < t_end) {
        __syncthreads();  // the previous tile's LDS reads are done
        stage(tile, masked);
        __syncthreads();
        const int nxt = next_open(tile + 1);
        const bool nxt_masked = nxt < t_end && tile_masked(nxt);
        if (nxt < t_end) issue(nxt, nxt_masked);
        // S^T = K Q^T for the tile's 64 positions and the wave's 16 rows:
        // lane (lg, l16) gets positions 16 t + 4 lg + i of row l16 (k steps
        // outer: four independent accumulations in flight)
        fm_f4 sc[4];
#pragma unroll
        for (int t = 0; t < 4; t++) sc[t] = fm_f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kk = 0; kk < KS; kk++) {
            fm_h8 kb[4];
#pragma unroll
            for (int t = 0; t < 4; t++) kb[t] = fm_load8(&s_k[16 * t + l16][32 * kk + 8 * lg]);
#pragma unroll
            for (int t = 0; t < 4; t++) sc[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kb[t], qa[kk], sc[t], 0, 0, 0);
        }
        // mask and online softmax of the lane's row: 16 of its 64 values in
        // the lane, the rest in lanes l16 + 16, + 32, + 48
        const int ql = (16 * wave + l16) / g;
        float sv[4][4], mx = -INFINITY;
        if (masked) {
#pragma unroll
            for (int t = 0; t < 4; t++) {
                const fm_f4 mk = *(const fm_f4 *) &s_m[ql][16 * t + 4 * lg];
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    sv[t][i] = mk[i] == -INFINITY ? -INFINITY : fmaf(sc[t][i], qscale, mk[i]);
                    mx = fmaxf(mx, sv[t][i]);
                }
            }
        } else {
#pragma unroll
            for (int t = 0; t < 4; t++)
#pragma unroll
                for (int i = 0; i < 4; i++) mx = fmaxf(mx, sc[t][i]);
            mx = mx * qscale;
        }
        mx = fmaxf(mx, __shfl_xor(mx, 16));
        mx = fmaxf(mx, __shfl_xor(mx, 32));
        const float mn = fmaxf(m, mx);
        const float base = mn == -INFINITY ? 0.0f : mn;  // a row with nothing open yet
        const float alpha = m == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m - base);
        // P^T in registers as the P V product's B operand: k slot 8 lg + j of
        // step kk holds position 32 kk + 16 (j / 4) + 4 lg + j % 4 -- this
        // lane's own values; V^T is read in the same order
        fm_h8 pb[kFmTile / 32];
        if (masked) {
#pragma unroll
            for (int t = 0; t < 4; t++)
#pragma unroll
                for (int i = 0; i < 4; i++)
                    pb[t >> 1][4 * (t & 1) + i] =
                        (_Float16) (sv[t][i] == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(sv[t][i] - base));
        } else {
#pragma unroll
            for (int t = 0; t < 4; t++)
#pragma unroll
                for (int i = 0; i < 4; i++)
                    pb[t >> 1][4 * (t & 1) + i] = (_Float16) __builtin_amdgcn_exp2f(fmaf(sc[t][i], qscale, -base));
        }
        // the row's sum of the f16 values: a product with ones, every lane of
        // the row's column gets it (32 VALU instructions and two cross-lane
        // steps a tile otherwise)
        fm_f4 ps = fm_f4{0.f, 0.f, 0.f, 0.f};
        const fm_h8 ones = {1, 1, 1, 1, 1, 1, 1, 1};
#pragma unroll
        for (int kk = 0; kk < kFmTile / 32; kk++) ps = __builtin_amdgcn_mfma_f32_16x16x32_f16(ones, pb[kk], ps, 0, 0, 0);
        l = l * alpha + ps[0];
        m = mn;
        // rescale the accumulators only when some row's maximum moved
        if (__any(alpha != 1.0f)) {
#pragma unroll
            for (int ct = 0; ct < NT; ct++) o[ct] *= alpha;
        }
        // O^T += V^T P^T: A lane (lg, l16) = dim 16 ct + l16 at the k slots'
        // positions, two 4-position runs of V^T
#pragma unroll
        for (int kk = 0; kk < kFmTile / 32; kk++) {
#pragma unroll
            for (int ct = 0; ct < NT; ct++) {
                const _Float16 * vrow = &s_vt[16 * ct + l16][32 * kk + 4 * lg];
                typedef _Float16 fm_h4 __attribute__((ext_vector_type(4)));
                const fm_h4 v0 = *(const fm_h4 *) vrow, v1 = *(const fm_h4 *) (vrow + 16);
                const fm_h8 va = {v0[0], v0[1], v0[2], v0[3], v1[0], v1[1], v1[2], v1[3]};
                o[ct] = __builtin_amdgcn_mfma_f32_16x16x32_f16(va, pb[kk], o[ct], 0, 0, 0);
            }
        }
        if constexpr (MG) {
            if (nxt >= z_end || nxt >= t_end) {
                // the split is done: merge its state, start the next one afresh
                float wa, wb;
                fm_merge(M, L, m, l, wa, wb);
#pragma unroll
                for (int ct = 0; ct < NT; ct++) {
                    O[ct] = O[ct] * wa + o[ct] * wb;
                    o[ct] = fm_f4{0.f, 0.f, 0.f, 0.f};
                }
                m = -INFINITY, l = 0.0f;
                while (z_end <= nxt) z_end += per;
            }
        }
        tile = nxt;
        masked = nxt_masked;
    }
    if (!MG && a.mfma_split > 1) {
        // partials of split z: O unnormalised, then (m, l), per workgroup row
        const int64_t blk = (int64_t) hs * q_blocks + qb;
        const int64_t all_rows = (int64_t) n_blk * kFmRows;
        const int64_t pr = (blk * a.mfma_split + z) * kFmRows + 16 * wave + l16;
#pragma unroll
        for (int ct = 0; ct < NT; ct++) *(fm_f4 *) &part[pr * D + 16 * ct + 4 * lg] = o[ct];
        if (lg == 0) {
            part[all_rows * D + 2 * pr] = m;
            part[all_rows * D + 2 * pr + 1] = l;
        }
        return;
    }
    // out = O / l, ggml's [D, hq, n_q, n_seq] layout
    const int r = 16 * wave + l16, i = q0 + r / g;
    if (i >= a.n_q) return;
    float * op = out + (((int64_t) seq * a.n_q + i) * a.hq + kvh * g + r % g) * D;
    const float inv = l > 0.0f ? 1.0f / l : 0.0f;
#pragma unroll
    for (int ct = 0; ct < NT; ct++) {
        fm_f4 v = fm_f4{0.f, 0.f, 0.f, 0.f};
        if constexpr (MG) {
            if (L > 0.0f) v = O[ct] / L;  // as the combine launch divides
        } else {
            v = o[ct] * inv;
        }
        *(fm_f4 *) &op[16 * ct + 4 * lg] = v;
    }
}

// the splits of a workgroup row merged in split order (fm_merge), then out =
// O / L (0 for a row with no live position). 256 threads: 256 / D rows, one
// dim a thread.
template <int D>
__global__ __launch_bounds__(kFmThreads) void k_fattn_mfma_combine(fattn_args a, const float * __restrict__ part,
                                                                   float * __restrict__ out, int q_blocks) {
    constexpr int RW = kFmThreads / D;
    const int dim = (int) threadIdx.x % D;
    const int64_t row = (int64_t) blockIdx.x * RW + (int) threadIdx.x / D;  // over blk * kFmRows
    const int64_t n_blk = (int64_t) q_blocks * a.hkv * a.n_seq;
    if (row >= n_blk * kFmRows) return;
    const int64_t blk = row / kFmRows;
    const int r = (int) (row % kFmRows);
    const int g = a.hq / a.hkv, qpw = kFmRows / g;
    const int bx = (int) (blk % q_blocks), by = (int) (blk / q_blocks);
    const int kvh = by % a.hkv, seq = by / a.hkv;
    const int i = bx * qpw + r / g, head = kvh * g + r % g;
    if (i >= a.n_q) return;
    const int ns = a.mfma_split;
    const int64_t all_rows = n_blk * ns * kFmRows;
    const float * ml = part + all_rows * D;
    // batches of kB splits: every load of a batch is requested before any is
    // used (indexes clamped to the last split, the extra terms masked), so a
    // batch costs one memory round trip
    constexpr int kB = 16;
    float M = -INFINITY, L = 0.0f, acc = 0.0f;
    for (int z0 = 0; z0 < ns; z0 += kB) {
        float mz[kB], lz[kB], oz[kB];
#pragma unroll
        for (int k = 0; k < kB; k++) {
            const int64_t pr = (blk * ns + min(z0 + k, ns - 1)) * kFmRows + r;
            mz[k] = ml[2 * pr];
            lz[k] = ml[2 * pr + 1];
            oz[k] = part[pr * D + dim];
        }
#pragma unroll
        for (int k = 0; k < kB; k++) {
            if (z0 + k >= ns) break;
            float wa, wb;
            fm_merge(M, L, mz[k], lz[k], wa, wb);
            acc = acc * wa + oz[k] * wb;
        }
    }
    out[(((int64_t) seq * a.n_q + i) * a.hq + head) * D + dim] = L > 0.0f ? acc / L : 0.0f;
}

static int fm_q_blocks(const fattn_args & a) {
    const int qpw = kFmRows / (a.hq / a.hkv);
    return (a.n_q + qpw - 1) / qpw;
}

// Whether the splits of a (planned over n_tiles tiles) are merged in the
// workgroup, by a model of both forms' times in units of T, the 2.0 us that one
// workgroup alone on a CU takes for a tile (at either head size). F(n) is the
// time in which the CUs, n workgroups dealt to them, do a tile of each: with
// heads of 128 two are resident and take 1.39 T, further ones come after them;
// with heads of 64 (three resident) two take 1.27 T, three 1.53 T, from four on
// 0.53 T each.
// Merged, there are `blocks` workgroups of the whole span; most spans have a
// masked tail, which these skip: 0.9 of it is counted. Split, there are
// blocks x splits, each of a part of the span (with heads of 64 they fill the
// CUs evenly), and the combine and the partials cost 6 T and, with heads of
// 128, 1/128 T a workgroup. With 64-wide heads the split form reads f32 K and V
// itself, the merged one copies of them (8 T). So merging is refused where few
// blocks over a long span would leave CUs idle; and below a block for every
// second CU, where the combine is small and costs less than the 6 T (one sequence
// over 512 positions, in a row without waits: 32 queries 16.9 / 22.0, 119 19.7 /
// 22.6, 256 22.8 / 22.3; 119 over 1000 of 1024 20.3 / 38.1).
// Measured, us a call, split / merged (128: 16 query, 8 kv heads; queries, live
// positions and span, sequences):
//   128 blocks  256 q 640 of 1024, 2     44 / 38    256 q 2000 of 2048, 2    60 / 80
//               256 q 1000 of 1024, 2    45 / 49    512 q 8000 of 8192, 1   114 / 253
//   192 blocks  256 q 1000 of 1024, 3    61 / 49    256 q 3000 of 4096, 3   106 / 113
//   256 blocks  256 q 1500 of 2048, 4    98 / 68    256 q 8000 of 8192, 4   210 / 256
//               512 q 3000 of 4096, 2   127 / 113   1024 q 4000 of 4096, 1  123 / 137
//   320 blocks  256 q 3000 of 4096, 5   162 / 146   256 q 8000 of 8192, 5   261 / 336
//   504 blocks  2000 q 4000 of 4096, 1  223 / 170
//   512 blocks  256 q 3000 of 4096, 8   256 / 148
//   576 blocks                                      288 q 8000 of 8192, 8   459 / 543
// Heads of 64 over f16 K and V, 6 heads: 256 q 500 of 512, 8 sequences (192
// blocks) 37 / 29, 1500 of 1500, 4 (576) 101 / 84, 1 (144) 45 / 59; over f32, 14
// heads: 600 of 600, 8 (1120) 117 / 112, 1300 of 1300, 1 (294) 71 / 84. The rule
// takes the slower form by up to 8 % at the edges (256 q 1000 of 1024, 2).
static bool fm_merge_pays(const fattn_args & a, int64_t blocks, int n_tiles, bool kv_f32, int n_cu) {
    if (2 * blocks < n_cu) return false;
    const bool wide = a.d == 128;
    auto shared = [&](int64_t n) {
        const double k = (double) ((n + n_cu - 1) / n_cu);
        return wide ? 1.39 * std::floor(k / 2) + std::fmod(k, 2.0) : std::max(0.53 * k, 0.75 + 0.26 * k);
    };
    const int64_t wgs = blocks * a.mfma_split;
    const double per = (double) ((n_tiles + a.mfma_split - 1) / a.mfma_split);
    const double merged = 0.9 * n_tiles * shared(blocks) + (kv_f32 && !wide ? 8.0 : 0.0);
    const double split = (wide ? per * shared(wgs) : 0.53 * n_tiles * (double) blocks / n_cu) + 6.0 + (double) (wgs * a.d) / 16384;
    return merged <= split;
}

void fattn_mfma_plan(fattn_args & a, int n_cu, bool kv_f32) {
    // split the span when one sequence's query blocks leave CUs idle: up to
    // two workgroups a CU (their LDS and registers fit twice), at least four
    // tiles a split. Planned from one sequence's shape, so a sequence's rows
    // get the same bits batched or alone.
    const int64_t base = (int64_t) fm_q_blocks(a) * a.hkv;
    const int n_tiles = (a.n_kv + kFmTile - 1) / kFmTile;
    int split = 1;
    if (base < 2 * n_cu) split = (int) std::min<int64_t>((2 * n_cu + base - 1) / base, std::max(1, n_tiles / 4));
    // a split covers at most kFmMaxSpan positions (its live bits in LDS)
    split = std::max(split, (n_tiles + kFmMaxSpan / kFmTile - 1) / (kFmMaxSpan / kFmTile));
    // no empty split: every split owns at least one tile
    const int per = (n_tiles + split - 1) / split;
    a.mfma_split = (n_tiles + per - 1) / per;
    // merged or split, the bits are the same
    a.mfma_merge = a.mfma_split > 1 && a.n_kv <= kFmMaxSpan && fm_merge_pays(a, base * a.n_seq, n_tiles, kv_f32, n_cu);
}

size_t fattn_mfma_scratch_bytes(const fattn_args & a) {
    if (a.mfma_split <= 1 || a.mfma_merge) return 0;
    const int64_t rows = (int64_t) fm_q_blocks(a) * a.hkv * a.n_seq * a.mfma_split * kFmRows;
    return (size_t) rows * (a.d + 2) * sizeof(float);
}

bool fattn_mfma_supported(const fattn_args & a) {
    const int g = a.hkv > 0 ? a.hq / a.hkv : 0;
    // K / V rows, heads and sequences start on 16 bytes (16-byte row loads)
    const bool aligned = (a.k_nb1 | a.k_nb2 | a.k_nb3 | a.v_nb1 | a.v_nb2 | a.v_nb3) % 16 == 0;
    // one mask row for every head (the planner's FLASH_ATTN_EXT contract)
    return (a.d == 64 || a.d == 128) && a.n_q > 1 && g >= 1 && g <= 8 && kFmRows % g == 0 && a.n_kv > 0 && aligned &&
           (!a.mask || a.m_ne2 == 1);
}

bool fattn_mfma_reads_f32(const fattn_args & a) {
    // the 64-wide heads of the encoders (the staging registers double)
    return a.mfma && a.d == 64 && !a.mfma_merge;
}

void launch_fattn_mfma(const fattn_args & a, void * scratch, float * out, hipStream_t s) {
    const int qb = fm_q_blocks(a);
    const bool merged = a.mfma_merge;
    const int64_t base = (int64_t) qb * a.hkv * a.n_seq;
    const dim3 grid((unsigned) (base * (merged ? 1 : a.mfma_split)));
    float * part = (float *) scratch;
    const uintptr_t mal = (uintptr_t) a.mask | (uintptr_t) a.m_nb1 | (uintptr_t) a.m_nb3;
    const int mm = !a.mask ? 0 : (mal & 15) == 0 ? 1 : (mal & 3) == 0 ? 3 : 2;
    auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, dim3(kFmThreads), 0, s, a, out, part); };
    auto form = [&](auto d, auto mg) {
        constexpr int D = decltype(d)::value;
        constexpr bool MG = decltype(mg)::value;
        if (mm == 0) go(k_fattn_mfma<D, 0, MG, false>);
        else if (mm == 1) go(k_fattn_mfma<D, 1, MG, false>);
        else if (mm == 3) go(k_fattn_mfma<D, 3, MG, false>);
        else go(k_fattn_mfma<D, 2, MG, false>);
    };
    using d128 = std::integral_constant<int, 128>;
    using d64 = std::integral_constant<int, 64>;
    if (a.mfma_kv32) {
        if (!fattn_mfma_reads_f32(a)) {
            note_hip_error(hipErrorInvalidValue);
            return;
        }
        if (mm == 0) go(k_fattn_mfma<64, 0, false, true>);
        else if (mm == 1) go(k_fattn_mfma<64, 1, false, true>);
        else if (mm == 3) go(k_fattn_mfma<64, 3, false, true>);
        else go(k_fattn_mfma<64, 2, false, true>);
    } else if (a.d == 128 && merged) form(d128{}, std::true_type{});
    else if (a.d == 128) form(d128{}, std::false_type{});
    else if (merged) form(d64{}, std::true_type{});
    else form(d64{}, std::false_type{});
    note_hip_error(hipGetLastError());
    if (a.mfma_split > 1 && !merged) {
        const int64_t rows = (int64_t) qb * a.hkv * a.n_seq * kFmRows;
        const int rw = kFmThreads / a.d;
        const unsigned wgs = (unsigned) ((rows + rw - 1) / rw);
        if (a.d == 128) hipLaunchKernelGGL(k_fattn_mfma_combine<128>, dim3(wgs), dim3(kFmThreads), 0, s, a, part, out, qb);
        else hipLaunchKernelGGL(k_fattn_mfma_combine<64>, dim3(wgs), dim3(kFmThreads), 0, s, a, part, out, qb);
        note_hip_error(hipGetLastError());
    }
}

}  // namespace mi355x
