// Partition kernels of the gfx950 decode library and their launchers, as
// templates: each partial_*.hip translation unit instantiates those of one q
// format and head dimension (decode.hip's run_partial picks the unit), so the
// library's many kernel instantiations compile in parallel.
#ifndef PAGED_DECODE_PARTITION_KERNELS_H
#define PAGED_DECODE_PARTITION_KERNELS_H

#include "device_common.h"

namespace pd {
// ---------------------------------------------------------------------------
// Partition kernels.
//
// Both kernels cut every partition of split_tokens tokens into kQuarters
// contiguous quarters and give each quarter of each KV head (and head tile) to
// one wave, which leaves its own max-corrected state per query head in the
// workspace: numerator [B, Hq, 4 * splits, D] and stats [B, Hq, 4 * splits, 2],
// state index 4 * split + quarter. Waves never combine with each other, so the
// kernels have no workgroup barrier on the hot path.


// A chunk's scores may exceed the running max by up to 2^kRescaleSlack before
// the accumulators are rescaled; weights then stay <= 2^8, far from overflow.
constexpr float kRescaleSlack = 8.0f;

// Stores one wave's state for its GT heads. acc[g][e] lives in the row layout
// (lanes [r*LPT, (r+1)*LPT) = token row r, dims col*EPL .. col*EPL+EPL-1) and
// has already been summed over rows into the lanes of row 0; m and l for head g
// are in lane g.
template <int D, int GT, int EPL, int LPT>
__device__ __forceinline__ void store_wave_state(const PartialParams& p, const WaveWork& w, int lane,
                                                 const float (&acc)[GT][EPL], float m, float l) {
    const int part = w.split * kQuarters + w.quarter;
    if (lane < LPT) {
        const int col = lane;
#pragma unroll
        for (int g = 0; g < GT; ++g) {
            if (g < w.heads_here) {
                f32x4* dst = reinterpret_cast<f32x4*>(p.numerator + numerator_offset(p, w.q_row + g, part, D) + col * EPL);
#pragma unroll
                for (int e = 0; e < EPL; e += 4)
                    dst[e / 4] = f32x4{acc[g][e], acc[g][e + 1], acc[g][e + 2], acc[g][e + 3]} * p.v_scale;
            }
        }
    }
    if (lane < w.heads_here) {
        float2* st = reinterpret_cast<float2*>(p.stats + stats_offset(p, w.q_row + lane, part));
        *st = make_float2(l > 0.0f ? m : kNoToken, l);
    }
}

// Empty states (m = -FLT_MAX, l = 0: an identity of every merge) for the
// wave's quarter of the `extra` live partitions after its first one, when a
// tail item streamed several partitions as one.
__device__ __forceinline__ void store_empty_states(const PartialParams& p, const WaveWork& w, int lane, int extra) {
    if (lane >= w.heads_here) return;
    for (int e = 1; e <= extra; ++e)
        *reinterpret_cast<float2*>(p.stats + stats_offset(p, w.q_row + lane, (w.split + e) * kQuarters + w.quarter)) =
            make_float2(kNoToken, 0.0f);
}

// ---------------------------------------------------------------------------
// FP32 partition kernel: both contractions on v_mfma_f32_4x4x1_16b_f32, whose
// products and sums are those of fmaf.
//
// A wave takes tiles of four tokens. K is loaded as lane (block = lane / 4,
// token = lane % 4), 16 bytes per lane: the MFMA's rows are the tile's tokens,
// its columns four query heads and its sixteen blocks sixteen slices of the
// dims, so each lane ends with four tokens' partial scores of head lane % 4.
// Summing them over the blocks also spreads the tokens (sum_scores): row group
// r of the lanes -- [r*LPT, (r+1)*LPT) -- keeps tokens r, r + TPL, ..., which is
// the A operand of P.V (rows = heads, blocks = dims), V being loaded in row
// layout: lanes of row group r hold token r of a TPL-token load, 16 bytes each.
// Every row group keeps its own online-softmax stream, head h's in the lanes
// with lane % 4 == h % 4; they are combined at the end of the wave.
//
// Per four FP32 tokens of D 128 with four heads: 16 MFMAs (8 cycles each) and
// about 45 other vector instructions. The vector ALU alone took about 200, with
// a 5-step sum over the lanes for each head and token and a softmax that every
// lane repeated, and waited for its loads at the end of each block of 32 tokens.
// A ring of R tiles stays in flight: the next K is requested once a tile is
// scored, the next V once it is summed; the range's last ring requests nothing
// and takes only the tiles that are there (MQA B49 of up to 33 tokens with D 64,
// us: 9.28 -> 7.88). Measured on
// MI355X (decode call, us, with the launch shape of plan_fp32; vector ALU ->
// this): B8 L4096 ragged, 158 MB 44.68 -> 35.66; uniform B2 L4096 23.96 ->
// 16.11, B16 116.93 -> 101.95;
// MHA B1 L16384 106.71 -> 88.46; D 64: GQA 8 B32 L3000 ragged 53.66 -> 34.95, MQA B64
// L2048 39.40 -> 25.06; whole rows B64 L256 35.18 -> 28.33.
// kRow: a whole-row workgroup (up to kRowMaxWaves waves) that folds its
// waves' states in LDS and writes the output rows instead of states.

__device__ __forceinline__ __amdgpu_buffer_rsrc_t tile_buffer(const char* base, uint32_t bytes);

// Sums of a 4-token score quadruple over the MFMA's blocks (lanes lane % 4
// apart): x[s] is token TPL * s + lane / LPT of the tile, in all lanes of its
// row group with the same lane % 4.
template <int LPT>
__device__ __forceinline__ void sum_scores(const f32x4& sc, float (&x)[LPT / 16]) {
    constexpr int kRowRor4 = 0x124, kRowRor8 = 0x128;
    if constexpr (LPT == 32) {
        x[0] = swap32_sum(sc[0], sc[1]);
        x[1] = swap32_sum(sc[2], sc[3]);
#pragma unroll
        for (int s = 0; s < 2; ++s) x[s] = swap16_sum(x[s], x[s]);
    } else {
        const float even = swap32_sum(sc[0], sc[2]), odd = swap32_sum(sc[1], sc[3]);
        x[0] = swap16_sum(even, odd);
    }
#pragma unroll
    for (int s = 0; s < LPT / 16; ++s) {
        x[s] += dpp_move<kRowRor4>(x[s]);
        x[s] += dpp_move<kRowRor8>(x[s]);
    }
}

// Lane 4 * (lane / 4) + kLane's value.
template <int kLane>
__device__ __forceinline__ float quad_lane(float x) {
    return dpp_move<kLane * 0x55>(x);
}

__device__ __forceinline__ float quad_lane(float x, int i) {
    return i == 0 ? quad_lane<0>(x) : i == 1 ? quad_lane<1>(x) : i == 2 ? quad_lane<2>(x) : quad_lane<3>(x);
}

template <int D, int GT, int R, bool kStreamV, int kList, bool kRow = false>
__global__ void __launch_bounds__(kRow ? kWave * fp32_row_max_waves(GT) : kWave * 8)
    partial_kernel(const PartialParams p) {
    constexpr int EPL = 4;
    constexpr int LPT = D / EPL;
    constexpr int TPL = kWave / LPT;
    constexpr int TT = kFp32TileTokens;
    constexpr int NL = TT / TPL;        // loads per tile of K, and of V
    constexpr int HG = (GT + 3) / 4;    // head groups of four
    static_assert(D == 64 * NL, "K loads of 64 dims");

    struct Tile {
        u32x4 k[NL];
        u32x4 v[NL];
    };
    struct Request {
        uint64_t base;
        uint32_t bytes;  // of the tile's live rows (0: nothing to read)
    };

    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int lane = threadIdx.x % kWave;
    const int row = lane / LPT;
    const int col = lane % LPT;
    const BlockCoords bc = block_coords<kList>(blockIdx.x, blockIdx.y, blockIdx.z, p.grid_x, p.grid_y, p.xcd_shift,
                                                     p.xcd_main_rows, p.xcd_tail_shift, p.head_shift);
    const PartitionRange pr = partition_range<kList>(p, bc);
    const int waves_wg = blockDim.x / kWave;
    const int32_t* pages = p.table + static_cast<int64_t>(pr.b) * p.table_width;
    int window = kRow ? row_speculative_page<TT>(p, wave, waves_wg)
                      : speculative_page<TT>(p, pr.first, pr.count, pr.qgroup, wave);
    int window_ids = pages[window_entry(p, window, lane)];
    const int len_raw = p.lengths[pr.b];
    const WaveWork w = kRow ? row_wave_work<GT, TT>(p, pr.b, bc.heads, wave, waves_wg, len_raw)
                            : wave_work<GT, TT>(p, pr.b, pr.first, pr.count, pr.qgroup, bc.heads, wave, len_raw);
    // Whole-row waves with an empty slice stay for the fold (empty state).
    if (!kRow && w.dead) {
        // Never read: the merge stops at the sequence's last live partition.
        // The speculative page-id window is consumed here (an empty asm
        // operand) so that its load is issued before this branch, alongside
        // the length's, rather than sunk into the live path after it.
        asm volatile("" ::"v"(window_ids));
        return;
    }
    const float* q_base = static_cast<const float*>(p.q) + w.q_row * D;

    // B operand of q.K^T: head 4 hg + lane % 4, dims 64 i + 4 (lane / 4) on.
    f32x4 qv[HG][NL];
#pragma unroll
    for (int hg = 0; hg < HG; ++hg) {
        const int head = 4 * hg + lane % 4;
#pragma unroll
        for (int i = 0; i < NL; ++i) {
            qv[hg][i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            if (head < w.heads_here)
                qv[hg][i] = *reinterpret_cast<const f32x4*>(q_base + head * D + 64 * i + 4 * (lane / 4));
        }
    }
    float m_head[HG], l_head[HG];  // of head 4 hg + lane % 4 and this lane's row group
    f32x4 sum[HG][EPL];            // sum[hg][e][r]: head 4 hg + r, dim col * EPL + e
#pragma unroll
    for (int hg = 0; hg < HG; ++hg) {
        m_head[hg] = kNoToken;
        l_head[hg] = 0.0f;
#pragma unroll
        for (int e = 0; e < EPL; ++e) sum[hg][e] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    }
    const char* k_head = static_cast<const char*>(p.k) + static_cast<size_t>(w.kv_head) * D * 4;
    const char* v_head = static_cast<const char*>(p.v) + static_cast<size_t>(w.kv_head) * D * 4;
    const uint32_t k_lane = tile_row_offset(p, lane % 4, static_cast<uint32_t>(lane / 4) * 16u);
    const uint32_t v_lane = tile_row_offset(p, row, static_cast<uint32_t>(col) * 16u);
    int rb = w.wb, re = w.wb;

    auto locate = [&](int t0) {
        const int page = __builtin_amdgcn_readlane(window_ids, tile_slot(p, t0, window));
        return Request{tile_base(p, page, t0), tile_bytes(p, tile_live(p, t0, re, page), t0, re, TT)};
    };
    auto load_k = [&](Tile& t, const Request& rq) {
        const __amdgpu_buffer_rsrc_t kb = tile_buffer(k_head + rq.base, rq.bytes);
#pragma unroll
        for (int i = 0; i < NL; ++i) t.k[i] = __builtin_amdgcn_raw_buffer_load_b128(kb, k_lane + 256u * i, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
    };
    auto load_v = [&](Tile& t, const Request& rq) {
        const __amdgpu_buffer_rsrc_t vb = tile_buffer(v_head + rq.base, rq.bytes);
#pragma unroll
        for (int i = 0; i < NL; ++i)
            t.v[i] = __builtin_amdgcn_raw_buffer_load_b128(vb, v_lane + tile_row_offset(p, TPL * i, 0), 0,
                                                           kStreamV ? 2 : 0);
        __builtin_amdgcn_sched_barrier(0);
    };

    auto score = [&](const Tile& t, float (&x)[HG][NL]) {
#pragma unroll
        for (int hg = 0; hg < HG; ++hg) {
            f32x4 sc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int i = 0; i < NL; ++i) {
                const f32x4 kf = __builtin_bit_cast(f32x4, t.k[i]);
#pragma unroll
                for (int e = 0; e < 4; ++e) sc = __builtin_amdgcn_mfma_f32_4x4x1f32(kf[e], qv[hg][i][e], sc, 0, 0, 0);
            }
            sum_scores<LPT>(sc, x[hg]);
        }
    };

    auto accumulate = [&](Tile& t, const Request& rq, float (&x)[HG][NL], int t0) {
        if (rq.bytes == 0u || t0 < rb || t0 + TT > re) {
#pragma unroll
            for (int s = 0; s < NL; ++s) {
                const int token = t0 + TPL * s + row;
                const bool valid = (rq.bytes != 0u) & (token >= rb) & (token < re);
#pragma unroll
                for (int hg = 0; hg < HG; ++hg) x[hg][s] = valid ? x[hg][s] : -INFINITY;
                // Rows before the range are another quarter's: their V stays out of this one's sums.
#pragma unroll
                for (int e = 0; e < 4; ++e) t.v[s][e] = token >= rb ? t.v[s][e] : 0u;
            }
        }
        float top[HG];
        bool grow = false;
#pragma unroll
        for (int hg = 0; hg < HG; ++hg) {
            top[hg] = x[hg][0];
#pragma unroll
            for (int s = 1; s < NL; ++s) top[hg] = fmaxf(top[hg], x[hg][s]);
            top[hg] *= p.scale_log2;
            grow |= top[hg] > m_head[hg] + kRescaleSlack;
        }
        if (__any(grow)) {
#pragma unroll
            for (int hg = 0; hg < HG; ++hg) {
                const float m_new = fmaxf(m_head[hg], top[hg]);
                const float alpha = fast_exp2(m_head[hg] - m_new);
                m_head[hg] = m_new;
                l_head[hg] *= alpha;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float a = quad_lane(alpha, r);
#pragma unroll
                    for (int e = 0; e < EPL; ++e) sum[hg][e][r] *= a;
                }
            }
        }
#pragma unroll
        for (int hg = 0; hg < HG; ++hg) {
#pragma unroll
            for (int s = 0; s < NL; ++s) {
                const float wt = fast_exp2(fmaf(x[hg][s], p.scale_log2, -m_head[hg]));
                l_head[hg] += wt;
                const f32x4 vf = __builtin_bit_cast(f32x4, t.v[s]);
#pragma unroll
                for (int e = 0; e < EPL; ++e)
                    sum[hg][e] = __builtin_amdgcn_mfma_f32_4x4x1f32(wt, vf[e], sum[hg][e], 0, 0, 0);
            }
        }
    };

    for (rb = w.wb; rb < w.we; rb = re) {
        if ((rb >> p.page_shift) != window) {
            window = rb >> p.page_shift;
            window_ids = pages[window_entry(p, window, lane)];
        }
        re = min(w.we, (window + kWave) << p.page_shift);
        Tile ring[R];
        Request at[R];
        int s0 = rb & ~(TT - 1);
#pragma unroll
        for (int c = 0; c < R; ++c) {
            at[c] = locate(s0 + c * TT);
            load_k(ring[c], at[c]);
            load_v(ring[c], at[c]);
        }
        for (; s0 + R * TT < re; s0 += R * TT) {
#pragma unroll
            for (int c = 0; c < R; ++c) {
                float x[HG][NL];
                score(ring[c], x);
                const Request next = locate(s0 + (R + c) * TT);
                load_k(ring[c], next);
                accumulate(ring[c], at[c], x, s0 + c * TT);
                load_v(ring[c], next);
                at[c] = next;
            }
        }
        // The last ring's tiles, as far as the range goes: nothing to request.
#pragma unroll
        for (int c = 0; c < R; ++c) {
            if (s0 + c * TT >= re) break;
            float x[HG][NL];
            score(ring[c], x);
            accumulate(ring[c], at[c], x, s0 + c * TT);
        }
    }

    // The row group's state with every head in every lane.
    float m[GT], l[GT], acc[GT][EPL];
#pragma unroll
    for (int g = 0; g < GT; ++g) {
        m[g] = quad_lane(m_head[g / 4], g % 4);
        l[g] = quad_lane(l_head[g / 4], g % 4);
#pragma unroll
        for (int e = 0; e < EPL; ++e) acc[g][e] = sum[g / 4][e][g % 4];
    }
    // Combine the TPL token-row streams (lanes LPT, 2*LPT, ... apart).
#pragma unroll
    for (int g = 0; g < GT; ++g) {
        float mw = m[g];
#pragma unroll
        for (int x = LPT; x < kWave; x <<= 1) mw = fmaxf(mw, __shfl_xor(mw, x));
        const float f = l[g] > 0.0f ? fast_exp2(m[g] - mw) : 0.0f;
        float lw = l[g] * f;
#pragma unroll
        for (int x = LPT; x < kWave; x <<= 1) lw += __shfl_xor(lw, x);
#pragma unroll
        for (int e = 0; e < EPL; ++e) {
            float a = acc[g][e] * f;
#pragma unroll
            for (int x = LPT; x < kWave; x <<= 1) a += __shfl_xor(a, x);
            acc[g][e] = a;
        }
        m[g] = mw;
        l[g] = lw;
    }
    if constexpr (kRow) {
        // Every wave leaves its state in its LDS slot -- m[8], l[8], then
        // acc[8][D] -- and after one barrier the workgroup forms each output
        // element of the tile's live heads as the merge does (max over the
        // states with l > 0, weights 2^(m - max), sum(weight * n) * v_scale /
        // sum(weight * l), or 0 for a row without tokens; decode.cu:94-107).
        extern __shared__ __attribute__((aligned(16))) float row_lds[];
        constexpr int kSlot = row_slot_bytes_fp32(D) / 4;
        float* slot = row_lds + wave * kSlot;
        if (lane == 0) {
#pragma unroll
            for (int g = 0; g < GT; ++g) {
                slot[g] = m[g];
                slot[8 + g] = l[g];
            }
        }
        if (lane < LPT) {
#pragma unroll
            for (int g = 0; g < GT; ++g)
#pragma unroll
                for (int e = 0; e < EPL; ++e) slot[16 + g * D + col * EPL + e] = acc[g][e];
        }
        __syncthreads();
        for (int o = threadIdx.x; o < w.heads_here * D; o += blockDim.x) {
            const int h = o / D;
            float mx = kNoToken;
            for (int s = 0; s < waves_wg; ++s) {
                const float* st = row_lds + s * kSlot;
                mx = st[8 + h] > 0.0f ? fmaxf(mx, st[h]) : mx;
            }
            float den = 0.0f, num = 0.0f;
            for (int s = 0; s < waves_wg; ++s) {
                const float* st = row_lds + s * kSlot;
                const float ls = st[8 + h];
                const float f = ls > 0.0f ? fast_exp2(st[h] - mx) : 0.0f;
                den = fmaf(f, ls, den);
                num = fmaf(f, st[16 + o], num);
            }
            p.out[w.q_row * D + o] = den > 0.0f ? num * p.v_scale / den : 0.0f;
        }
        return;
    }
    // Lane g needs head g's (m, l): every lane holds every head's values.
    float m_lane = m[0], l_lane = l[0];
#pragma unroll
    for (int g = 1; g < GT; ++g) {
        m_lane = lane == g ? m[g] : m_lane;
        l_lane = lane == g ? l[g] : l_lane;
    }
    store_wave_state<D, GT, EPL, LPT>(p, w, lane, acc, m_lane, l_lane);
    store_empty_states(p, w, lane, extra_live_partitions(p, pr.first, pr.count, len_raw));
}

// ---------------------------------------------------------------------------
// 16-bit partition kernel (q in FP16 or BF16; K/V in the same type or in FP8):
// q.K^T and P.V both on the matrix cores.
//
// A 16-token tile is scored with D/32 v_mfma_f32_16x16x32_{f16,bf16}: K in the
// A layout (lane l holds 8 consecutive dims, [32 s + 8 (l / 16), +8) of k-step
// s, of tile token sigma(l % 16)), q in the B layout (lane l: query head
// l % 16, zero past the group). K is loaded as whole token rows (16 bytes per
// lane, full cache lines, like V) and reaches the A layout through a per-wave
// LDS tile. With sigma(r) = r / 4 + 4 (r % 4) the result leaves lane l with
// head n = l % 16 and tokens g, g + 4, g + 8, g + 12 of the tile (g = l / 16).
// Tiles go in pairs: the scores of both are the A operand of
// v_mfma_f32_16x16x32 for P (row = head, k = 8 g + 4 h + e <-> token g + 4 e of
// tile h), so the weights never leave their lanes. V is loaded in the row
// layout -- load e covers tokens 4 e .. 4 e + 3, lanes [16 r, 16 r + 16) token
// 4 e + r, VH consecutive dims per lane -- so lane (g, n) holds tokens g + 4 e
// of dims n VH .. n VH + VH - 1, and element j of a pair's eight V loads is the
// B operand of MFMA block j (column n <-> dim n VH + j). P is split into high
// and low parts of the compute type (two MFMAs per block), which keeps the
// weights exact to about 2^-22 (FP16) or 2^-17 (BF16) relative. Each (head,
// dim) sum lives in exactly one lane: lane (g, n) ends with heads 4 g ..
// 4 g + 3 of dims n VH .. n VH + VH - 1, stored directly. One running max per
// head is shared by the wave, with lazy rescaling as in the FP32 kernel.
//
// What bounds it is the time a wave does not have loads in flight. With the
// waves of a grid all started together, blocks of loads followed by their
// computation left the memory idle while every wave computed: FP8 B16 L4096
// (ragged, 90 MB) ran 26 us where a plain gather of as many pages takes 15. So
// a pair's K is requested again (the next pair's) as soon as it is scored and
// its V as soon as it is summed; the descriptors' range check (tile_buffer)
// replaces clamped addresses, the softmax runs once per pair, and P.V takes
// 32 tokens per MFMA: about 115 vector instructions per 32 FP16 tokens, 370
// before. Measured on MI355X, decode call, us (graph, K/V rotated past the
// Infinity Cache; blocks of two or four tiles, FP8 -> pairs): FP8 B16 L4096
// ragged 33.1 -> 25.3, B32 51.4 -> 39.5, B64 L8192 164.6 -> 143.2, B4 L4096 15.6 ->
// 14.0; FP16 B1 L4096 10.2 -> 9.3, B4 18.1 -> 17.7, B8 ragged 22.9 -> 21.3, B16
// ragged 39.5 -> 36.7; FP16 MQA B256 L2048 31.6 -> 28.2; B64 L8192 ragged 231 ->
// 227. Two pairs in flight per wave (173 VGPRs and more, two waves per SIMD)
// were slower: FP8 B4 15.3, FP16 B4 18.7, B16 ragged FP8 27.8 against 26.9.
// Short ranges have nothing to overlap: a whole-row slice of one tile is read and
// scored alone, with P.V over its 16 tokens, an empty second tile is not scored,
// and a range's last pair requests nothing. Against pairs throughout (FP16, us):
// 640 rows of up to 64 tokens with D 128 9.05 -> 7.36, 1088 rows of 32 7.66 ->
// 6.08, MQA B256 of 256 tokens with D 64 10.14 -> 8.03, B16 of 640 tokens at split
// 128 with twice the context reserved 16.6 -> 16.0; the copy of the computation
// that this takes costs waves of two pairs up to 1.5% (64 / 8 heads B6 L4096 with
// twice the context reserved 26.3 -> 26.7).
//
// FP8 K/V (OCP e4m3 or e5m2) are loaded as bytes and converted to the compute
// type after they arrive; both formats convert exactly. The per-tensor scales
// cost nothing per element: k_scale is folded into the softmax scale and
// v_scale into the stored numerator.

enum KvFormat { kKvNative = 0, kKvE4M3 = 1, kKvE5M2 = 2 };


// Buffer descriptor of `bytes` bytes at base (uniform over the wave): loads
// from byte offset `bytes` on return zeros and touch no memory.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t tile_buffer(const char* base, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(base), 0, bytes, 0x00027000);
}

// N stored words at byte offset `offset` of a buffer. kStream marks 16-byte
// loads non-temporal (see plan_mfma for when that is used).
template <int N, bool kStream>
__device__ __forceinline__ void load_words(__amdgpu_buffer_rsrc_t buffer, uint32_t offset, uint32_t (&w)[N]) {
    constexpr int kAux = kStream && N == 4 ? 2 : 0;
    if constexpr (N == 4) {
        const u32x4 x = __builtin_amdgcn_raw_buffer_load_b128(buffer, offset, 0, kAux);
        w[0] = x[0];
        w[1] = x[1];
        w[2] = x[2];
        w[3] = x[3];
    } else if constexpr (N == 2) {
        const u32x2 x = __builtin_amdgcn_raw_buffer_load_b64(buffer, offset, 0, kAux);
        w[0] = x[0];
        w[1] = x[1];
    } else {
        w[0] = __builtin_amdgcn_raw_buffer_load_b32(buffer, offset, 0, kAux);
    }
}

// Matrix-core operations and conversions of one 16-bit compute type.
template <typename QT>
struct Compute;

template <>
struct Compute<_Float16> {
    static __device__ __forceinline__ f32x4 qk(const u32x4& a, const u32x4& b, const f32x4& c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0,
                                                      0, 0);
    }
    static __device__ __forceinline__ f32x4 pv(const u32x2& a, const u32x2& b, const f32x4& c) {
        return __builtin_amdgcn_mfma_f32_16x16x16f16(__builtin_bit_cast(f16x4, a), __builtin_bit_cast(f16x4, b), c, 0,
                                                     0, 0);
    }
    // Nearest 16-bit values of (a, b), packed, and those values back as FP32.
    static __device__ __forceinline__ uint32_t round(float a, float b, float& back_a, float& back_b) {
        const f16x2 h = __builtin_convertvector((f32x2{a, b}), f16x2);
        back_a = static_cast<float>(h[0]);
        back_b = static_cast<float>(h[1]);
        return __builtin_bit_cast(uint32_t, h);
    }
    // Bytes 2 HIGH, 2 HIGH + 1 of an FP8 word as a packed pair (exact).
    template <int KVF, bool HIGH>
    static __device__ __forceinline__ uint32_t from_fp8(uint32_t word) {
        f16x2 h;
        if constexpr (KVF == kKvE4M3) h = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(word, 1.0f, HIGH);
        else h = __builtin_amdgcn_cvt_scalef32_pk_f16_bf8(word, 1.0f, HIGH);
        return __builtin_bit_cast(uint32_t, h);
    }
};

template <>
struct Compute<__bf16> {
    static __device__ __forceinline__ f32x4 qk(const u32x4& a, const u32x4& b, const f32x4& c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c,
                                                       0, 0, 0);
    }
    static __device__ __forceinline__ f32x4 pv(const u32x2& a, const u32x2& b, const f32x4& c) {
        return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(s16x4, a), __builtin_bit_cast(s16x4, b), c,
                                                         0, 0, 0);
    }
    static __device__ __forceinline__ uint32_t round(float a, float b, float& back_a, float& back_b) {
        const bf16x2 h = __builtin_convertvector((f32x2{a, b}), bf16x2);
        const uint32_t bits = __builtin_bit_cast(uint32_t, h);
        back_a = __builtin_bit_cast(float, bits << 16);
        back_b = __builtin_bit_cast(float, bits & 0xFFFF0000u);
        return bits;
    }
    template <int KVF, bool HIGH>
    static __device__ __forceinline__ uint32_t from_fp8(uint32_t word) {
        f32x2 f;
        if constexpr (KVF == kKvE4M3) f = __builtin_amdgcn_cvt_pk_f32_fp8(word, HIGH);
        else f = __builtin_amdgcn_cvt_pk_f32_bf8(word, HIGH);
        const float f0 = f[0], f1 = f[1];  // FP8 values are exact in BF16: keep the top halves
        return (__builtin_bit_cast(uint32_t, f0) >> 16) | (__builtin_bit_cast(uint32_t, f1) & 0xFFFF0000u);
    }
};

// N stored words of K or V as compute-type pairs (2 N words for FP8).
template <typename QT, int KVF, int N>
__device__ __forceinline__ void to_compute(const uint32_t (&raw)[N], uint32_t (&out)[KVF == kKvNative ? N : 2 * N]) {
    if constexpr (KVF == kKvNative) {
#pragma unroll
        for (int i = 0; i < N; ++i) out[i] = raw[i];
    } else {
#pragma unroll
        for (int i = 0; i < N; ++i) {
            out[2 * i] = Compute<QT>::template from_fp8<KVF, false>(raw[i]);
            out[2 * i + 1] = Compute<QT>::template from_fp8<KVF, true>(raw[i]);
        }
    }
}

// Element j of each of the four V loads (VH elements per load, as VH / 2
// packed words), packed as an MFMA operand (k = load index).
template <int VH>
__device__ __forceinline__ u32x2 v_operand(const uint32_t (&v)[4][VH / 2], int j) {
    constexpr uint32_t kLow = 0x05040100u, kHigh = 0x07060302u;  // halves of (second, first)
    const uint32_t sel = j % 2 == 0 ? kLow : kHigh;
    return u32x2{__builtin_amdgcn_perm(v[1][j / 2], v[0][j / 2], sel),
                 __builtin_amdgcn_perm(v[3][j / 2], v[2][j / 2], sel)};
}

// LDS slot of the quarter combine: one quarter's state of one (KV head,
// head tile) -- per-head max and denominator, and the accumulator in the
// lanes' own layout (acc[j] of lane l at acc[j][l]).
template <int VH>
struct CombineSlot {
    float m[16];
    float l[16];
    f32x4 acc[VH][kWave];
};

// kStream: which 16-byte loads are non-temporal (see plan_mfma):
// 0 none, 1 V (and FP8 K, whose V loads are 8-byte), 2 K and V.
// kFold: what the workgroup stores -- 0 one state per wave; 1 one state per
// qw quarters of a partition (quarter combine); 2 the output rows of a whole
// row's states (whole-row launch, up to kRowMaxWaves waves: 1024 lanes).
//
// The waves per SIMD are those that the registers allow without a spill: left to
// itself the compiler takes 5 to 16 more for D 64 (FP16, 5 KV heads B32 L3000 with
// twice the context reserved: 22.6 -> 20.8 us).
constexpr int mfma_waves_per_simd(int head_dim, int elem) { return head_dim == 64 ? 5 : elem == 2 ? 3 : 4; }

template <typename QT, int KVF, int D, int GT, int kStream, int kFold, int kList>
__global__ void __launch_bounds__(kFold == 2 ? kWave * row_max_waves(D) : kWave * 8,
                                  mfma_waves_per_simd(D, KVF == kKvNative ? 2 : 1))
    partial_mfma_kernel(const PartialParams p) {
    using C = Compute<QT>;
    constexpr int ES = KVF == kKvNative ? 2 : 1;  // stored bytes per K/V element
    constexpr int KS = D / 32;                    // q.K^T k-steps (K loads) per tile
    constexpr int VH = D / 16;                    // V elements per lane per load = P.V MFMA blocks
    constexpr int VI = 4;                         // V loads per tile
    constexpr int VW = VH * ES / 4;               // stored words per V load
    static_assert(GT <= 16, "one MFMA column block holds at most 16 query heads");
    constexpr int kPair = 2;
    constexpr bool kLastApart = last_pair_apart(kList, ES);
    constexpr int kPairTokens = kPair * kTileTokens;

    // K is loaded whole rows at a time (KR lanes x 16 bytes per token, TK
    // tokens per load, KL loads per tile) and turned into the q.K^T operand
    // layout through a per-wave LDS tile. Its rows are padded by the size of
    // one operand read (16 bytes for 16-bit K, 8 for FP8), so the transposed
    // reads of 16 different rows fall in distinct banks.
    constexpr bool kStreamK = kStream == 2 || (kStream == 1 && KVF != kKvNative);
    constexpr int KR = D * ES / 16;
    constexpr int TK = kWave / KR;
    constexpr int KL = kTileTokens / TK;
    constexpr int kStageRow = mfma_stage_bytes(D, ES) / kTileTokens;
    static_assert(TK <= kTileTokens && kTileTokens % TK == 0, "whole row loads per tile");
    // Dynamic LDS: the waves' K tiles, then the quarter-combine slots
    // ([waves / qw][qw - 1] CombineSlot<VH>, kFold 1) or one slot per wave
    // (kFold 2); sized by the launch.
    extern __shared__ __attribute__((aligned(16))) char lds[];
    char* const k_stage = lds;
    char* const combine_lds = lds + mfma_stage_bytes(D, ES) * (blockDim.x / kWave);

    // Tiles are read and scored kPair at a time: one softmax step, and P.V
    // over all their tokens in one 16x16x32 MFMA per block.
    struct Request {  // where a pair of tiles lies
        uint64_t base[kPair];
        uint32_t bytes[kPair];  // of each tile's live rows (0: nothing to read)
    };
    struct Pair {
        uint32_t k[kPair][KL][4];
        uint32_t v[kPair][VI][VW];
    };

    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int lane = threadIdx.x % kWave;
    const int n = lane % 16;  // head (q.K^T, P) / column (P.V)
    const int g = lane / 16;  // lane group: tokens g + 4 e
    const BlockCoords bc = block_coords<kList>(blockIdx.x, blockIdx.y, blockIdx.z, p.grid_x, p.grid_y, p.xcd_shift,
                                                     p.xcd_main_rows, p.xcd_tail_shift, p.head_shift);
    const PartitionRange pr = partition_range<kList>(p, bc);
    // A whole-row workgroup's wave runs slice `wave` of its row (one KV head,
    // one head tile); otherwise the wave index splits into (head, tile,
    // quarter) within the workgroup's partition.
    const int waves_wg = blockDim.x / kWave;
    // The item's page-table row (a shared-prefix item's: its members' leader,
    // which its shared pass reads for every member that maps the same pages).
    const int32_t* pages = p.table + static_cast<int64_t>(pr.row) * p.table_width;
    int window = kFold == 2 ? row_speculative_page<kTileTokens>(p, wave, waves_wg)
                            : speculative_page<kTileTokens>(p, pr.first, pr.count, pr.qgroup, wave);
    int window_ids = pages[window_entry(p, window, lane)];
    // Members of a shared-prefix item (work lists only): lane m < members
    // holds member m's sequence and length; the wave covers the longest
    // member's tokens, and tile column n belongs to member n / GT, which
    // masks it at its own length. Any other item is one member, all columns.
    const bool grouped = kList == kGridList && pr.members > 1;
    int member_b = pr.b;
    int member_len = 0;
    int len_raw;
    if (grouped) {
        const bool is_member = lane < pr.members;
        member_b = p.prefix_order[pr.member0 + (is_member ? lane : 0)];
        member_len = is_member ? p.lengths[member_b] : 0;
        int longest = member_len;
#pragma unroll
        for (int offset = 8; offset > 0; offset >>= 1) longest = max(longest, __shfl_xor(longest, offset));
        len_raw = __builtin_amdgcn_readfirstlane(longest);
    } else {
        len_raw = p.lengths[pr.b];
    }
    const WaveWork w = kFold == 2 ? row_wave_work<GT, kTileTokens>(p, pr.b, bc.heads, wave, waves_wg, len_raw)
                                  : wave_work<GT, kTileTokens>(p, pr.b, pr.first, pr.count, pr.qgroup, bc.heads, wave,
                                                               len_raw);
    // A whole-row workgroup's waves with an empty slice stay to contribute
    // the empty state to the fold.
    if (kFold != 2 && w.dead) {
        // Never read: the merge stops at the sequence's last live partition.
        // The speculative page-id window is consumed here (an empty asm
        // operand) so that its load is issued before this branch, alongside
        // the length's, rather than sunk into the live path after it.
        asm volatile("" ::"v"(window_ids));
        return;
    }
    const char* q_row = static_cast<const char*>(p.q) + w.q_row * D * 2;
    // Column n's member, its query head within the tile, and its first masked
    // token: for a single-member item, member 0, head n, no mask of its own.
    const int col_slots = grouped ? GT : 16;
    const int col_member = n / col_slots;
    const int col_head = n - col_member * col_slots;
    const bool col_live = col_member < pr.members && col_head < w.heads_here;
    const int64_t row_base = static_cast<int64_t>(w.kv_head) * p.group + static_cast<int64_t>(w.tile) * GT;
    // q row (batch x query-head index) of member m's tile head 0.
    auto member_row = [&](int m) {
        return grouped ? static_cast<int64_t>(__shfl(member_b, m)) * p.query_heads + row_base : w.q_row;
    };
    // Formed again where it is used: kept, it would be spilled by the FP8 kernels
    // of shared-prefix items. (All lanes together: it reads other lanes.)
    auto col_row = [&] { return member_row(col_member) + col_head; };
    const int col_end = grouped ? min(max(__shfl(member_len, col_member), 0), p.reach) : 0x7FFFFFFF;

    // Page check of a shared-prefix item (prefix_span_pages): bit m of `own`
    // marks member m, whose table row differs from the leader's on a page
    // where it has tokens; it reads its own row in a later pass.
    uint32_t own = 0;
    if (grouped) {
        const int span = prefix_span_pages(p, w.wb, w.we);
        const int pairs = span * pr.members;
        uint32_t differs = 0;
        for (int base = 0; base < pairs; base += kWave) {
            const int pair = base + lane;
            const int m = pair < pairs ? prefix_pair_member(pair, span) : 0;
            const int page = prefix_pair_page(p, w.wb, pair < pairs ? pair : 0, span);
            const int mb = __shfl(member_b, m);
            const int m_end = min(min(max(__shfl(member_len, m), 0), p.reach), w.we);
            if (pair < pairs && (page << p.page_shift) < m_end &&
                p.table[static_cast<int64_t>(mb) * p.table_width + page] != pages[page])
                differs |= 1u << m;
        }
#pragma unroll
        for (int offset = 32; offset > 0; offset >>= 1) differs |= __shfl_xor(differs, offset);
        own = __builtin_amdgcn_readfirstlane(differs);
    }

    u32x4 qb[KS];
#pragma unroll
    for (int s = 0; s < KS; ++s) {
        qb[s] = u32x4{0u, 0u, 0u, 0u};
        if (grouped) {
            const int64_t row = col_row();
            if (col_live)
                qb[s] = *reinterpret_cast<const u32x4*>(static_cast<const char*>(p.q) +
                                                        (row * D + 32 * s + 8 * g) * 2);
        } else if (n < w.heads_here) {
            qb[s] = *reinterpret_cast<const u32x4*>(q_row + (n * D + 32 * s + 8 * g) * 2);
        }
    }

    float m_head = kNoToken;  // running max (log2 units) of head n, equal in all lane groups
    float l_part = 0.0f;      // this lane's share of head n's denominator
    f32x4 acc[VH];            // acc[j][i]: head 4 g + i, dim n VH + j
#pragma unroll
    for (int j = 0; j < VH; ++j) acc[j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    const char* k_head = static_cast<const char*>(p.k) + static_cast<size_t>(w.kv_head) * D * ES;
    const char* v_head = static_cast<const char*>(p.v) + static_cast<size_t>(w.kv_head) * D * ES;
    // This lane's bytes of row 0 of a tile's first K load and first V load.
    const uint32_t k_lane = tile_row_offset(p, lane / KR, static_cast<uint32_t>(lane % KR) * 16u);
    const uint32_t v_lane = tile_row_offset(p, g, static_cast<uint32_t>(n) * VH * ES);
    const int k_row_token = k_token_of_row(n);
    int rb = w.wb, re = w.wb;
    // The pass: its page-table row, its token end, and whether this lane's
    // column takes part (the shared pass: every member but those in `own`).
    const int32_t* pass_pages = pages;
    int pass_end = w.we;
    bool col_on = !grouped || ((own >> col_member) & 1u) == 0;

    auto locate = [&](int t0) {
        Request rq;
#pragma unroll
        for (int h = 0; h < kPair; ++h) {
            const int t = t0 + h * kTileTokens;
            const int page = __builtin_amdgcn_readlane(window_ids, tile_slot(p, t, window));
            rq.base[h] = tile_base(p, page, t);
            rq.bytes[h] = tile_bytes(p, tile_live(p, t, re, page), t, re);
        }
        return rq;
    };
    // The next three take the tiles of a request that are used: kPair, or the
    // first alone.
    auto load_k = [&](auto tiles, Pair& pr2, const Request& rq) {
#pragma unroll
        for (int h = 0; h < decltype(tiles)::value; ++h) {
            const __amdgpu_buffer_rsrc_t kb = tile_buffer(k_head + rq.base[h], rq.bytes[h]);
#pragma unroll
            for (int s = 0; s < KL; ++s)
                load_words<4, kStreamK>(kb, k_lane + tile_row_offset(p, TK * s, 0), pr2.k[h][s]);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    auto load_v = [&](auto tiles, Pair& pr2, const Request& rq) {
#pragma unroll
        for (int h = 0; h < decltype(tiles)::value; ++h) {
            const __amdgpu_buffer_rsrc_t vb = tile_buffer(v_head + rq.base[h], rq.bytes[h]);
#pragma unroll
            for (int e = 0; e < VI; ++e)
                load_words<VW, (kStream >= 1)>(vb, v_lane + tile_row_offset(p, 4 * e, 0), pr2.v[h][e]);
        }
        __builtin_amdgcn_sched_barrier(0);
    };

    // Raw scores of tile h of the pair at t0: K through the wave's LDS tile
    // into the operand layout, then q.K^T.
    auto score = [&](const Pair& pr2, int h) {
        f32x4 sc = {0.0f, 0.0f, 0.0f, 0.0f};
        char* stage = k_stage + wave * (kTileTokens * kStageRow);
        __builtin_amdgcn_wave_barrier();  // the previous tile's reads are issued before these writes
#pragma unroll
        for (int s = 0; s < KL; ++s) {
            const uint32_t* kw = pr2.k[h][s];
            char* dst = stage + (TK * s + lane / KR) * kStageRow + (lane % KR) * 16;
            if constexpr (kStageRow % 16 == 0) {
                *reinterpret_cast<u32x4*>(dst) = u32x4{kw[0], kw[1], kw[2], kw[3]};
            } else {  // FP8 rows are 8-byte aligned
                reinterpret_cast<u32x2*>(dst)[0] = u32x2{kw[0], kw[1]};
                reinterpret_cast<u32x2*>(dst)[1] = u32x2{kw[2], kw[3]};
            }
        }
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            const char* src = stage + k_row_token * kStageRow + (32 * s + 8 * g) * ES;
            if constexpr (KVF == kKvNative) {
                sc = C::qk(*reinterpret_cast<const u32x4*>(src), qb[s], sc);
            } else {
                const u32x2 raw2 = *reinterpret_cast<const u32x2*>(src);
                const uint32_t raw[2] = {raw2[0], raw2[1]};
                uint32_t kq[4];
                to_compute<QT, KVF, 2>(raw, kq);
                sc = C::qk(u32x4{kq[0], kq[1], kq[2], kq[3]}, qb[s], sc);
            }
        }
        return sc;
    };

    // Softmax and P.V of the tiles at t0, whose scores are sc.
    auto accumulate = [&](auto tiles, Pair& pr2, const Request& rq, f32x4 (&sc)[kPair], int t0) {
        constexpr int NT = decltype(tiles)::value;
        float mx = -INFINITY;
#pragma unroll
        for (int h = 0; h < NT; ++h) {
            const int t1 = t0 + h * kTileTokens;
            // Whole tiles of an ungrouped item need no mask.
            if (grouped || rq.bytes[h] == 0u || t1 < rb || t1 + kTileTokens > re) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int t = t1 + g + 4 * e;
                    const bool valid = (rq.bytes[h] != 0u) & (t >= rb) & (t < re) & (t < col_end) & col_on;
                    sc[h][e] = valid ? sc[h][e] : -INFINITY;
                    // Rows before the range are another quarter's: their V stays out of this one's sums.
#pragma unroll
                    for (int i = 0; i < VW; ++i) pr2.v[h][e][i] = t >= rb ? pr2.v[h][e][i] : 0u;
                }
            }
            mx = fmaxf(mx, fmaxf(fmaxf(sc[h][0], sc[h][1]), fmaxf(sc[h][2], sc[h][3])));
        }
        const float pair_max = max_over_lane_groups(mx) * p.scale_log2;
        if (__builtin_amdgcn_ballot_w64((n < GT * pr.members) & (pair_max > m_head + kRescaleSlack)) != 0) {
            const float m_new = fmaxf(m_head, pair_max);
            const float alpha = fast_exp2(m_head - m_new);
            m_head = m_new;
            l_part *= alpha;
            // acc[.][i] belongs to head 4 g + i, whose factor lives in lane 4 g + i.
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float a = __shfl(alpha, 4 * g + i);
#pragma unroll
                for (int j = 0; j < VH; ++j) acc[j][i] *= a;
            }
        }
        // P in high and low parts, k = 8 g + 4 h + e <-> token g + 4 e of tile h.
        u32x4 p_hi{}, p_lo{};
#pragma unroll
        for (int h = 0; h < NT; ++h) {
#pragma unroll
            for (int e = 0; e < 4; e += 2) {
                const float w0 = fast_exp2(fmaf(sc[h][e], p.scale_log2, -m_head));
                const float w1 = fast_exp2(fmaf(sc[h][e + 1], p.scale_log2, -m_head));
                l_part += w0;
                l_part += w1;
                float back0, back1, unused0, unused1;
                p_hi[2 * h + e / 2] = C::round(w0, w1, back0, back1);
                p_lo[2 * h + e / 2] = C::round(w0 - back0, w1 - back1, unused0, unused1);
            }
        }
        // One stored word of every V load at a time, so that only its converted
        // form is live (FP8: the words of 4 of the lane's dims become 8 of them).
        constexpr int kWordDims = 4 / ES;
#pragma unroll
        for (int w4 = 0; w4 < VW; ++w4) {
            uint32_t vq[NT][VI][kWordDims / 2];
#pragma unroll
            for (int h = 0; h < NT; ++h)
#pragma unroll
                for (int e = 0; e < VI; ++e) {
                    const uint32_t raw[1] = {pr2.v[h][e][w4]};
                    to_compute<QT, KVF, 1>(raw, vq[h][e]);
                }
#pragma unroll
            for (int j = 0; j < kWordDims; ++j) {
                const u32x2 v0 = v_operand<kWordDims>(vq[0], j);
                f32x4& sum = acc[w4 * kWordDims + j];
                if constexpr (NT == 1) {
                    sum = C::pv(u32x2{p_hi[0], p_hi[1]}, v0, sum);
                    sum = C::pv(u32x2{p_lo[0], p_lo[1]}, v0, sum);
                } else {
                    const u32x2 v1 = v_operand<kWordDims>(vq[1], j);
                    const u32x4 vo = {v0[0], v0[1], v1[0], v1[1]};
                    sum = C::qk(p_hi, vo, sum);
                    sum = C::qk(p_lo, vo, sum);
                }
            }
            if constexpr (KVF != kKvNative) __builtin_amdgcn_sched_barrier(0);
        }
    };

    constexpr std::integral_constant<int, 1> one{};
    constexpr std::integral_constant<int, kPair> two{};
    uint32_t pending = own;
    if (kFold == 2 && one_tile_slice(w)) {
        // A whole-row slice of one tile at most (short rows).
        if (w.wb < w.we) {
            if ((w.wb >> p.page_shift) != window) {
                window = w.wb >> p.page_shift;
                window_ids = pages[window_entry(p, window, lane)];
            }
            re = w.we;
            Pair pair;
            const Request at = locate(w.wb);
            load_k(one, pair, at);
            load_v(one, pair, at);
            f32x4 sc[kPair];
            sc[0] = score(pair, 0);
            accumulate(one, pair, at, sc, w.wb);
        }
    } else for (;;) {
        for (rb = w.wb; rb < pass_end; rb = re) {
            if ((rb >> p.page_shift) != window) {
                window = rb >> p.page_shift;
                window_ids = pass_pages[window_entry(p, window, lane)];
            }
            re = min(pass_end, (window + kWave) << p.page_shift);
            // Once a pair's K is scored, the next pair's is requested into its
            // registers, and likewise V, so that loads are in flight while the
            // wave computes. The range's last pair, which requests nothing, is
            // outside the loop (kLastApart): the compiler then counts the loads
            // outstanding at every wait, as it could not past a request that is
            // skipped.
            int t0 = rb & ~(kTileTokens - 1);
            Pair pair;
            Request at = locate(t0);
            load_k(two, pair, at);
            load_v(two, pair, at);
            f32x4 sc[kPair];
            for (; t0 + (kLastApart ? kPairTokens : 0) < re; t0 += kPairTokens) {
#pragma unroll
                for (int h = 0; h < kPair; ++h) sc[h] = score(pair, h);
                const Request next = locate(t0 + kPairTokens);
                load_k(two, pair, next);
                accumulate(two, pair, at, sc, t0);
                load_v(two, pair, next);
                at = next;
            }
            if constexpr (kLastApart) {
                sc[0] = score(pair, 0);
                sc[1] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
                if (at.bytes[1] != 0u) sc[1] = score(pair, 1);
                accumulate(two, pair, at, sc, t0);
            }
        }
        if (!grouped || pending == 0) break;
        // Next member with a row of its own: its row, up to its own end.
        const int m = __builtin_ctz(pending);
        pending &= pending - 1;
        const int b = __builtin_amdgcn_readlane(member_b, m);
        pass_pages = p.table + static_cast<int64_t>(b) * p.table_width;
        pass_end = min(w.we, min(max(p.lengths[b], 0), p.reach));
        col_on = col_member == m;
        window = -1;
    }

    // Lane (g, n) holds heads 4 g + i of dims n VH .. n VH + VH - 1; the
    // denominator of head n is summed over the four lane groups.
    float l_head = sum_over_lane_groups(l_part);
    if constexpr (kFold == 2) {
        // Every wave leaves its state in its slot; after one barrier the
        // workgroup forms each output element of the tile's live heads as the
        // merge does: the max over the states with l > 0, their weights
        // 2^(m - max), and sum(weight * n) * v_scale / sum(weight * l), or 0
        // for a row without tokens (decode.cu:94-107). Thread o covers
        // elements o, o + blockDim.x, ...: column n of dims n VH + j, head h,
        // with n fastest, so a slot's accumulators are read in lane order.
        CombineSlot<VH>* slots = reinterpret_cast<CombineSlot<VH>*>(combine_lds);
        CombineSlot<VH>* mine = slots + wave;
        if (lane < 16) {
            mine->m[n] = m_head;
            mine->l[n] = l_head;
        }
#pragma unroll
        for (int j = 0; j < VH; ++j) mine->acc[j][lane] = acc[j];
        __syncthreads();
        const int waves = waves_wg;
        for (int o = threadIdx.x; o < w.heads_here * D; o += blockDim.x) {
            const int col = o % 16;
            const int j = (o / 16) % VH;
            const int h = o / D;
            const int src_lane = 16 * (h / 4) + col;
            float mx = kNoToken;
            for (int s = 0; s < waves; ++s) mx = slots[s].l[h] > 0.0f ? fmaxf(mx, slots[s].m[h]) : mx;
            float den = 0.0f, num = 0.0f;
            for (int s = 0; s < waves; ++s) {
                const float ls = slots[s].l[h];
                const float f = ls > 0.0f ? fast_exp2(slots[s].m[h] - mx) : 0.0f;
                den = fmaf(f, ls, den);
                num = fmaf(f, slots[s].acc[j][src_lane][h % 4], num);
            }
            p.out[(w.q_row + h) * D + col * VH + j] = den > 0.0f ? num * p.v_scale / den : 0.0f;
        }
        return;
    }
    const int part = w.split * kQuarters + w.quarter;
    if (!grouped) store_empty_states(p, w, lane, extra_live_partitions(p, pr.first, pr.count, len_raw));
    // A member whose own length ends before the partition (shorter on the
    // device than its host bound) stores nothing, like a dead item: no state
    // past a sequence's end is written. Column h's end lives in lane h.
    const int64_t part_first = static_cast<int64_t>(w.split) * p.split_tokens;
    auto column_alive = [&](int h) { return !grouped || part_first < __shfl(col_end, h); };
    if constexpr (kFold == 1) {
        // The workgroup's qw quarters of one (KV head, head tile) -- waves
        // wave - wave % qw onwards, all of one partition, so all live or all
        // gone above -- become one state: quarters 1 .. qw - 1 leave theirs in
        // LDS, and after one barrier the first quarter folds them into its own
        // in quarter order (the merge's max-corrected sum) and stores the
        // result. The other quarters' slots get the empty state (l = 0), which
        // every merge of the four-states-per-partition layout reads as an
        // identity.
        const int qw = p.quarters_per_wg;
        const int qq = wave % qw;
        CombineSlot<VH>* slots = reinterpret_cast<CombineSlot<VH>*>(combine_lds) + wave / qw * (qw - 1);
        if (qq != 0) {
            CombineSlot<VH>* slot = slots + (qq - 1);
            if (lane < 16) {
                slot->m[n] = m_head;
                slot->l[n] = l_head;
            }
#pragma unroll
            for (int j = 0; j < VH; ++j) slot->acc[j][lane] = acc[j];
            const int64_t row = col_row();
            if (lane < 16 && col_live && part_first < col_end)
                *reinterpret_cast<float2*>(p.stats + stats_offset(p, row, part)) = make_float2(kNoToken, 0.0f);
        }
        __syncthreads();
        if (qq != 0) return;
        for (int s = 0; s < qw - 1; ++s) {
            const CombineSlot<VH>* slot = slots + s;
            f32x4 in[VH];
#pragma unroll
            for (int j = 0; j < VH; ++j) in[j] = slot->acc[j][lane];
            const float m_in = slot->m[n];
            const float m_new = fmaxf(m_head, m_in);
            const float f_in = fast_exp2(m_in - m_new);  // 0 for an empty state, 1 if both are empty
            const float f_own = fast_exp2(m_head - m_new);
            l_head = fmaf(f_in, slot->l[n], f_own * l_head);
            m_head = m_new;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float a_in = __shfl(f_in, 4 * g + i);  // factors of head 4 g + i
                const float a_own = __shfl(f_own, 4 * g + i);
#pragma unroll
                for (int j = 0; j < VH; ++j) acc[j][i] = fmaf(a_in, in[j][i], a_own * acc[j][i]);
            }
        }
    }
    // acc[.][i] is tile column h = 4 g + i: member h / col_slots, head h % col_slots.
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int h = 4 * g + i;
        const int m = h / col_slots;
        const int hm = h - m * col_slots;
        const int64_t row = member_row(m) + hm;
        const bool alive = column_alive(h);
        if (m < pr.members && hm < w.heads_here && alive) {
            f32x4* dst = reinterpret_cast<f32x4*>(p.numerator + numerator_offset(p, row, part, D) + n * VH);
#pragma unroll
            for (int j = 0; j < VH; j += 4)
                dst[j / 4] = f32x4{acc[j][i], acc[j + 1][i], acc[j + 2][i], acc[j + 3][i]} * p.v_scale;
        }
    }
    const int64_t row = col_row();
    if (lane < 16 && col_live && part_first < col_end) {
        float2* st = reinterpret_cast<float2*>(p.stats + stats_offset(p, row, part));
        *st = make_float2(l_head > 0.0f ? m_head : kNoToken, l_head);
    }
}

inline int launch_status() { return hipGetLastError() == hipSuccess ? PD_OK : PD_ERR_LAUNCH; }

// Compute units of the current device, read once per device.
inline int device_compute_units() {
    static std::atomic<int> cached[64];
    int device = 0;
    if (hipGetDevice(&device) != hipSuccess || device < 0 || device >= 64) return 256;
    int cus = cached[device].load(std::memory_order_relaxed);
    if (cus == 0) {
        if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess || cus <= 0)
            cus = 256;  // MI355X
        cached[device].store(cus, std::memory_order_relaxed);
    }
    return cus;
}

inline dim3 to_dim3(const Grid& g) { return dim3(g.x, g.y, g.z); }

// Launches the matrix-core kernel planned by plan_mfma (head tile GT, stream
// mode and quarter combine chosen there).
template <typename QT, int KVF, int D, int GT>
int launch_mfma(const PartialParams& prm, int kv_heads, hipStream_t stream) {
    static_assert(sizeof(CombineSlot<D / 16>) == 2 * 16 * 4 + (D / 16) * kWave * 16, "combine_slot_bytes");
    const dim3 grid = to_dim3(partial_grid(prm, kv_heads));
    const dim3 block(partial_threads(prm));
    const size_t lds = static_cast<size_t>(mfma_lds_bytes(prm, D, KVF == kKvNative ? 2 : 1));
    const int kind = grid_kind(prm);
    // Whole-row launches are rectangular (one workgroup per row).
#define PD_LAUNCH_MFMA(MODE, FOLD)                                                                                \
    do {                                                                                                          \
        if constexpr (FOLD == 2)                                                                                  \
            hipLaunchKernelGGL((partial_mfma_kernel<QT, KVF, D, GT, MODE, 2, kGridRect>), \
                               grid, block, lds, stream, prm);                                                    \
        else if (kind == kGridList)                                                                               \
            hipLaunchKernelGGL((partial_mfma_kernel<QT, KVF, D, GT, MODE, FOLD, kGridList>), grid,      \
                               block, lds, stream, prm);                                                          \
        else if (kind == kGridRectTails)                                                                          \
            hipLaunchKernelGGL((partial_mfma_kernel<QT, KVF, D, GT, MODE, FOLD, kGridRectTails>), grid, \
                               block, lds, stream, prm);                                                          \
        else                                                                                                      \
            hipLaunchKernelGGL((partial_mfma_kernel<QT, KVF, D, GT, MODE, FOLD, kGridRect>), grid,      \
                               block, lds, stream, prm);                                                          \
    } while (0)
#define PD_LAUNCH_MFMA_FOLDS(MODE)                      \
    do {                                                \
        if (prm.row_mode) PD_LAUNCH_MFMA(MODE, 2);      \
        else if (prm.combine) PD_LAUNCH_MFMA(MODE, 1);  \
        else PD_LAUNCH_MFMA(MODE, 0);                   \
    } while (0)
    if constexpr (KVF == kKvNative) {
        if (prm.stream_mode == 2) {
            PD_LAUNCH_MFMA_FOLDS(2);
            return launch_status();
        }
    }
    if (prm.stream_mode >= 1) PD_LAUNCH_MFMA_FOLDS(1);
    else PD_LAUNCH_MFMA_FOLDS(0);
#undef PD_LAUNCH_MFMA_FOLDS
#undef PD_LAUNCH_MFMA
    return launch_status();
}

template <int D, int GT>
int launch_fp32(const PartialParams& prm, int kv_heads, hipStream_t stream) {
    const dim3 grid = to_dim3(partial_grid(prm, kv_heads));
    const dim3 block(partial_threads(prm));
    const int kind = grid_kind(prm);
#define PD_LAUNCH_FP32(STREAM)                                                                                      \
    do {                                                                                                            \
        if (kind == kGridList)                                                                                      \
            hipLaunchKernelGGL((partial_kernel<D, GT, kFp32Ring, STREAM, kGridList>), grid, block, 0, stream, prm); \
        else if (kind == kGridRectTails)                                                                            \
            hipLaunchKernelGGL((partial_kernel<D, GT, kFp32Ring, STREAM, kGridRectTails>), grid, block, 0, stream,  \
                               prm);                                                                                \
        else                                                                                                        \
            hipLaunchKernelGGL((partial_kernel<D, GT, kFp32Ring, STREAM, kGridRect>), grid, block, 0, stream, prm); \
    } while (0)
    if (prm.row_mode)
        hipLaunchKernelGGL((partial_kernel<D, GT, kFp32RowRing, false, kGridRect, true>), grid, block,
                           static_cast<size_t>(prm.row_waves) * row_slot_bytes_fp32(D), stream, prm);
    else if (prm.stream_mode != 0)
        PD_LAUNCH_FP32(true);
    else
        PD_LAUNCH_FP32(false);
#undef PD_LAUNCH_FP32
    return launch_status();
}

template <typename QT, int KVF, int D>
int dispatch_mfma(PartialParams& prm, int kv_heads, hipStream_t stream) {
    plan_mfma(prm, kv_heads, device_compute_units(), D, KVF == kKvNative ? 2 : 1);
    switch (prm.head_tile) {
        case 1: return launch_mfma<QT, KVF, D, 1>(prm, kv_heads, stream);
        case 2: return launch_mfma<QT, KVF, D, 2>(prm, kv_heads, stream);
        case 4: return launch_mfma<QT, KVF, D, 4>(prm, kv_heads, stream);
        case 8: return launch_mfma<QT, KVF, D, 8>(prm, kv_heads, stream);
        default: return launch_mfma<QT, KVF, D, 16>(prm, kv_heads, stream);
    }
}

template <int D>
int dispatch_fp32(PartialParams& prm, int kv_heads, hipStream_t stream) {
    plan_fp32(prm, kv_heads, D, device_compute_units());
    switch (prm.head_tile) {
        case 1: return launch_fp32<D, 1>(prm, kv_heads, stream);
        case 2: return launch_fp32<D, 2>(prm, kv_heads, stream);
        case 4: return launch_fp32<D, 4>(prm, kv_heads, stream);
        default: return launch_fp32<D, 8>(prm, kv_heads, stream);
    }
}

template <typename QT, int D>
int dispatch_kv(PartialParams& prm, int kv_dtype, int kv_heads, hipStream_t stream) {
    switch (kv_dtype) {
        case PD_DTYPE_FP8_E4M3: return dispatch_mfma<QT, kKvE4M3, D>(prm, kv_heads, stream);
        case PD_DTYPE_FP8_E5M2: return dispatch_mfma<QT, kKvE5M2, D>(prm, kv_heads, stream);
        default: return dispatch_mfma<QT, kKvNative, D>(prm, kv_heads, stream);
    }
}

// Launch the partition kernel of one (q format, head dimension), planned from
// prm (whose shape fields are set): one definition per partial_*.hip unit.
int dispatch_partial_f32_d64(PartialParams& prm, int kv_dtype, int kv_heads, hipStream_t stream);
int dispatch_partial_f32_d128(PartialParams& prm, int kv_dtype, int kv_heads, hipStream_t stream);
int dispatch_partial_f16_d64(PartialParams& prm, int kv_dtype, int kv_heads, hipStream_t stream);
int dispatch_partial_f16_d128(PartialParams& prm, int kv_dtype, int kv_heads, hipStream_t stream);
int dispatch_partial_bf16_d64(PartialParams& prm, int kv_dtype, int kv_heads, hipStream_t stream);
int dispatch_partial_bf16_d128(PartialParams& prm, int kv_dtype, int kv_heads, hipStream_t stream);

}  // namespace pd

#endif  // PAGED_DECODE_PARTITION_KERNELS_H
