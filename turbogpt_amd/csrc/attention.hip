// Causal softmax attention for gfx950, head_dim 64: flash-style forward (online softmax, fp32
// log-sum-exp saved) and recompute backward.  Takes the slot of attention_forward /
// attention_backward in the reference's layer (cuda/attention.cuh:48-106; called from
// cuda/model.cuh:20 and :86-88); the packed [token][q|k|v] buffer and the [token][head*64+d]
// output keep the reference's layout (cuda/attention.cuh:38-39,68), so no permutes are needed.
//
// All kernels work on 32x32 MFMA tiles (v_mfma_f32_32x32x16_bf16) and are written in the
// "transposed" form: the score tile is produced as S^T[key][query] so that one lane owns one
// query row - row maxima / sums / rescales are per-lane scalars - and the fp32 accumulator
// registers of S^T can be fed back, converted to bf16, as the B operand of the next product with
// no cross-lane movement.  The operand that must then be read "k-strided" (V for P.V, K for dS.K,
// Q and dO for the dK/dV products) is fetched with the transposing LDS read ds_read_b64_tr_b16.
//
// backward = two launches: dQ (one block per 128 queries, loops over key tiles; it also computes
// delta = rowsum(dO o O) for its queries), then dK/dV (one block per 128 keys, loops over query
// tiles).  No atomics: every output element has one owner and a fixed summation order, so results
// are bit-reproducible.
//
// Where 128-row blocks would leave the chip part idle (few or short sequences), blocks of 32 rows take their place,
// whose four waves share out the tiles of the reduced side: attn_fwd_split_kernel, and attn_bwd_split_kernel for the
// whole backward in one launch; between those sizes and the large ones the two backward kernels run side by side
// (forward_splits and backward_way have the rules).
#include "common.h"
#include <algorithm>
#include <atomic>
#include "../../include/tgk_kernels.h"

namespace {

constexpr int HD = 64;      // head dimension
constexpr float LOG2E = 1.4426950408889634f, LN2 = 0.6931471805599453f;

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef short s16x8 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;

TG_DEVICE f32x16 zero16() {
    f32x16 z;
#pragma unroll
    for (int r = 0; r < 16; ++r)
        z[r] = 0.f;
    return z;
}
TG_DEVICE f32x16 mfma(bf16x8 rows_to_regs, bf16x8 rows_to_lanes, f32x16 acc) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(rows_to_regs, rows_to_lanes, acc, 0, 0, 0);
}
// row index owned by accumulator register r of a 32x32 tile (lane half g = lane/32)
TG_DEVICE int acc_row(int r, int g) {
    return 8 * (r >> 2) + 4 * g + (r & 3);
}
// registers 8*kk2 .. 8*kk2+7 of an fp32 accumulator as a bf16 operand fragment
TG_DEVICE bf16x8 acc_to_frag(const f32x16 &acc, int kk2) {
    bf16x8 f;
#pragma unroll
    for (int j = 0; j < 8; ++j)
        f[j] = (__bf16)acc[8 * kk2 + j];
    return f;
}
TG_DEVICE float exp2_fast(float x) {
    return __builtin_amdgcn_exp2f(x);
}

// ---- swizzled 64 x 64 LDS tiles filled by wave-wide global -> LDS copies -------------------------
// 128-byte rows, no padding (a copy fills 1 KiB contiguously); the 16-byte chunk c of row r sits at
// chunk c ^ swz(r).  swz is chosen so that both access patterns are bank-conflict free: fragments along
// the rows (16 consecutive rows, one chunk each) and transposing reads along the columns (4 consecutive
// rows, 32 bytes each).
constexpr int TILE_ELEMS = 64 * 64;
TG_DEVICE int swz(int row) {
    return (((row >> 1) & 1) << 2) | ((row >> 2) & 3);
}
// this wave's two copies (regions wave and wave+4, 8 rows each) of a 64-row tile starting at `base`
TG_DEVICE void tile_copy_async_one(uint32_t lds_tile, const bf16_t *base, int ld, int wave, int lane, int j) {
    const int region = wave + 4 * j, row = region * 8 + (lane >> 3), chunk = (lane & 7) ^ swz(row);
    async_copy16(__builtin_amdgcn_readfirstlane(lds_tile + region * 1024), base + size_t(row) * ld + chunk * 8);
}
// byte offset of this lane's 16 bytes within a 64-row tile whose rows are ld elements apart
TG_DEVICE uint32_t tile_copy_offset(int ld, int wave, int lane, int j) {
    const int region = wave + 4 * j, row = region * 8 + (lane >> 3), chunk = (lane & 7) ^ swz(row);
    return uint32_t(row * ld + chunk * 8) * 2;
}
TG_DEVICE void tile_copy_async(uint32_t lds_tile, const bf16_t *base, int ld, int wave, int lane) {
#pragma unroll
    for (int j = 0; j < 2; ++j)
        tile_copy_async_one(lds_tile, base, ld, wave, lane, j);
}
// The swizzle terms of both fragment kinds depend on the lane only (swz(row + 32) = swz(row);
// swz(r + 16) = swz(r)), so a kernel computes these element offsets once and adds compile-time
// constants per k-step / tile inside its loops.
// operand fragment along the rows: row mt*32 + lane%32, k = ks*16 + 8*(lane/32) .. +7
struct RowFragOffsets {
    int at[4];
    TG_DEVICE explicit RowFragOffsets(int lane) {
        const int row = lane & 31;
#pragma unroll
        for (int ks = 0; ks < 4; ++ks)
            at[ks] = row * 64 + (((ks * 2 + (lane >> 5)) ^ swz(row)) << 3);
    }
    TG_DEVICE bf16x8 load(const bf16_t *tile, int mt, int ks) const {
        return *reinterpret_cast<const bf16x8 *>(tile + at[ks] + mt * 32 * 64);
    }
};
// operand fragment along the columns (transposing reads): column dt*32 + lane%32 and the 8 rows
// kk*16 + 4g + {0..3}, kk*16 + 8 + 4g + {0..3} - the rows that accumulator registers 8*(kk%2) .. +7 of a
// 32x32 tile hold (acc_row), so a converted accumulator and this fragment agree on the reduced index
struct ColFragOffsets {
    int lo[2], hi[2];
    TG_DEVICE explicit ColFragOffsets(int lane) {
        const int g = lane >> 5, blk = (lane >> 4) & 1, i = lane & 15;
        const int r = 4 * g + (i >> 2);
#pragma unroll
        for (int dt = 0; dt < 2; ++dt) {
            const int col = dt * 32 + 16 * blk + 4 * (i & 3);
            lo[dt] = r * 64 + (((col >> 3) ^ swz(r)) << 3) + (col & 7);
            hi[dt] = (r + 8) * 64 + (((col >> 3) ^ swz(r + 8)) << 3) + (col & 7);
        }
    }
    TG_DEVICE bf16x8 load(const bf16_t *tile, int kk, int dt) const {
        const s16x4 a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4 *)(tile + lo[dt] + kk * 16 * 64));
        const s16x4 b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4 *)(tile + hi[dt] + kk * 16 * 64));
        const s16x8 both = __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7);
        return __builtin_bit_cast(bf16x8, both);
    }
};

// Block placement.  The work of a causal tile grows with its index and consecutive block ids go to the
// eight XCDs in turn, so a (tile, head, batch) grid whose tile extent is a multiple of 8 hands one XCD
// all the heaviest tiles.  Instead each XCD takes every eighth (batch, head) pair with all of that
// pair's tiles - which also keeps a pair's keys and values in one L2 - heaviest rank first.  The last `dealt` pairs
// are dealt out tile by tile instead, ahead of the others.
struct CausalBlock {
    int rank, h, b;
    bool live;
};
struct CausalGrid {
    int H, pairs, ranks, dealt;
    TG_DEVICE CausalBlock block(unsigned index) const {
        const int xcd = index & 7, slot = index >> 3, whole = pairs - dealt, per_xcd = (whole + 7) >> 3;
        const int deals = (dealt * ranks + 7) >> 3; // slots of an XCD that take tiles of the dealt pairs
        int rank, pair;
        if (slot < deals) {
            const int tile = slot * 8 + xcd;
            rank = tile / dealt;
            pair = whole + tile % dealt;
            return {rank, pair % H, pair / H, rank < ranks};
        }
        rank = (slot - deals) / per_xcd;
        pair = (slot - deals) % per_xcd * 8 + xcd;
        return {rank, pair % H, pair / H, pair < whole};
    }
    unsigned blocks() const {
        return (unsigned(dealt * ranks + 7) / 8 + unsigned((pairs - dealt + 7) / 8) * unsigned(ranks)) * 8;
    }
};
// Where eight does not divide the pairs, whole pairs give some XCDs a pair more than others, or leave some idle.  Dealing
// the remainder costs every XCD its own copy of those pairs' keys and values, so it is done only where the fullest XCD
// has more blocks than compute units.  Whole -> dealt, 128-row blocks, forward; backward in us: 1 pair of 8192 106 -> 98;
// 298 -> 274, 9 pairs of 8192 144 -> 123; 401 -> 329, 13 pairs of 8192 170 -> 160; 479 -> 444; but 15 pairs of 2048 (32
// blocks an XCD) 28.7 -> 32.5; 76 -> 79.  32-row blocks: 12 pairs of 1024 8.9 -> 8.6; 26.5 -> 20.3, 4 pairs of 4096
// 33 -> 20; 114 -> 58.
// The forward's 128-row blocks are short enough for the copies to outweigh that below 64 blocks a pair: whole -> dealt us, 4096
// positions 13 pairs 58.3 -> 62.2, 30 pairs 83.3 -> 89.5, 1920 and 2048 30 pairs 30.1 -> 31.3 and 32.2 -> 33.3; 8192 20 pairs 219 -> 200.
CausalGrid causal_grid(int B, int H, int T, int rows, int least_ranks = 1) {
    const int pairs = B * H, ranks = T / rows;
    return {H, pairs, ranks, (pairs + 7) / 8 * ranks > 32 && ranks >= least_ranks ? pairs % 8 : 0};
}

template <int N> struct Const {
    static constexpr int value = N;
};
// Lanes i and i+32 own the two halves of one query's keys.  v_permlane32_swap of a value with itself
// leaves the lower lanes' values in every lane of the first result and the upper lanes' in the second.
TG_DEVICE float halves_max(float x) {
    const auto both = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return fmaxf(__uint_as_float(both[0]), __uint_as_float(both[1]));
}
TG_DEVICE float halves_sum(float x) {
    const auto both = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float(both[0]) + __uint_as_float(both[1]);
}
// Writes a 32 x 32 accumulator whose rows (lane % 32) are rows of memory: `row` points at this lane's row, first
// of the 32 columns.  Lane l holds columns 8*q4 + 4*g + {0..3} (registers 4*q4 ..) of its row, lane l + 32 the
// other four of every eight.  The two trade halves, so that one ends up with columns 0..15 and the other with
// 16..31 and each writes 32 contiguous bytes: a quarter of the store instructions and of the cache lines touched
// per instruction that 8-byte pieces take.
TG_DEVICE void store_acc_rows(bf16_t *row, const f32x16 &acc, float scale, int g) {
    uint32_t x[4], y[4];
#pragma unroll
    for (int q4 = 0; q4 < 4; ++q4) {
        x[q4] = pack_bf16(acc[q4 * 4 + 0] * scale, acc[q4 * 4 + 1] * scale);
        y[q4] = pack_bf16(acc[q4 * 4 + 2] * scale, acc[q4 * 4 + 3] * scale);
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const auto ax = __builtin_amdgcn_permlane32_swap(x[h], x[h + 2], false, false);
        const auto ay = __builtin_amdgcn_permlane32_swap(y[h], y[h + 2], false, false);
        *reinterpret_cast<u32x4 *>(row + 16 * g + 8 * h) = u32x4{ax[0], ay[0], ax[1], ay[1]};
    }
}

// ---- one wave, one 64-row tile: the arithmetic of the three kernels ------------------------------------------
// forward, S^T: scores of 64 keys against 32 queries (lane % 32)
TG_DEVICE void scores(const bf16_t *kt, const RowFragOffsets &krows, const bf16x8 (&qf)[4], f32x16 (&s)[2]) {
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
#pragma unroll
        for (int mt = 0; mt < 2; ++mt)
            s[mt] = mfma(krows.load(kt, mt, ks), qf[ks], ks == 0 ? zero16() : s[mt]);
}
// forward: the scores of keys kv0 .. kv0 + 63 to probabilities under the running maximum m; l is this lane's half of
// the keys only, the halves are joined at the end.  Returns what earlier sums have to be multiplied by.
// ANY_TILE: the first tile seen need not be the row's first, so its scores may all be -inf (products that overflow) where
// the row has others: they get probability 0 and the maximum stays -inf.
template <bool ANY_TILE>
TG_DEVICE float online_softmax(f32x16 (&s)[2], int kv0, int wave_q0, int qrow, int g, float c, float &m, float &l) {
    if (kv0 + 63 > wave_q0) { // diagonal tile: hide keys after the query
#pragma unroll
        for (int mt = 0; mt < 2; ++mt)
#pragma unroll
            for (int r = 0; r < 16; ++r)
                if (kv0 + mt * 32 + acc_row(r, g) > qrow)
                    s[mt][r] = -INFINITY;
    }
    float mx = -INFINITY;
#pragma unroll
    for (int mt = 0; mt < 2; ++mt)
#pragma unroll
        for (int r = 0; r < 16; ++r)
            mx = fmaxf(mx, s[mt][r]);
    mx = halves_max(mx);
    const float m_new = fmaxf(m, mx * c);
    const float shift = ANY_TILE && m_new == -INFINITY ? 0.f : m_new;
    const float alpha = exp2_fast(m - shift);
    float sum = 0.f;
#pragma unroll
    for (int mt = 0; mt < 2; ++mt)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const float p = exp2_fast(fmaf(s[mt][r], c, -shift));
            s[mt][r] = p;
            sum += p;
        }
    l = l * alpha + sum;
    m = m_new;
    return alpha;
}
// forward: O^T += V^T P of the same 64 keys
TG_DEVICE void weigh_values(const bf16_t *vt, const ColFragOffsets &vcols, const f32x16 (&s)[2], f32x16 (&o)[2]) {
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
        const bf16x8 pf = acc_to_frag(s[kk >> 1], kk & 1);
#pragma unroll
        for (int dt = 0; dt < 2; ++dt)
            o[dt] = mfma(vcols.load(vt, kk, dt), pf, o[dt]);
    }
}
// dQ of 32 queries from 64 keys, in 32-key halves to keep the registers down
TG_DEVICE void dq_tile(const bf16_t *kt, const bf16_t *vt, int kv0, int wave_q0, int qrow, int g, float c, float lse,
                       const RowFragOffsets &krows, const ColFragOffsets &kcols, const bf16x8 (&qf)[4], const bf16x8 (&gf)[4],
                       const f32x16 &minus_delta, f32x16 (&dq)[2]) {
    const bool diagonal = kv0 + 63 > wave_q0;
#pragma unroll
    for (int mt = 0; mt < 2; ++mt) {
        if (kv0 + mt * 32 > wave_q0 + 31) // every key of this half follows this wave's queries
            continue;
        // dP - delta in one go: the product accumulates onto a register set that holds -delta of this lane's query
        f32x16 s = zero16(), dp;
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
            s = mfma(krows.load(kt, mt, ks), qf[ks], s);
            dp = mfma(krows.load(vt, mt, ks), gf[ks], ks == 0 ? minus_delta : dp);
        }
        // the causal mask only in the tiles that straddle the diagonal (wave-uniform branch)
        auto probabilities = [&](auto masked) {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                float p = exp2_fast(fmaf(s[r], c, -lse));
                if (decltype(masked)::value && kv0 + mt * 32 + acc_row(r, g) > qrow)
                    p = 0.f;
                dp[r] = p * dp[r];
            }
        };
        if (diagonal)
            probabilities(Const<1>{});
        else
            probabilities(Const<0>{});
#pragma unroll
        for (int kk2 = 0; kk2 < 2; ++kk2) {
            const bf16x8 dsf = acc_to_frag(dp, kk2);
#pragma unroll
            for (int dt = 0; dt < 2; ++dt)
                dq[dt] = mfma(kcols.load(kt, mt * 2 + kk2, dt), dsf, dq[dt]);
        }
    }
}
// dK, dV of 32 keys from 64 queries (from q0), in 32-query halves; `lse2` and `minus` in LDS: the queries' base-2
// log-sum-exps and negated deltas
TG_DEVICE void dkdv_tile(const bf16_t *qt_tile, const bf16_t *gt_tile, const float *lse2, const float *minus, int q0, int wave_k0,
                         int krow, int g, float c, const RowFragOffsets &qrows, const ColFragOffsets &qcols,
                         const bf16x8 (&kf)[4], const bf16x8 (&vf)[4], f32x16 (&dk)[2], f32x16 (&dv)[2]) {
    auto half = [&](auto half_tag) {
        constexpr int qt = decltype(half_tag)::value;
        const int qh = q0 + qt * 32;
        if (qh + 31 < wave_k0) // every query of this half precedes this wave's keys (wave uniform)
            return;
        // dP - delta in one go: the product accumulates onto -delta of its rows (the dQ kernel leaves the deltas
        // negated), one subtraction per score less on the vector ALU that bounds this kernel
        f32x16 s = zero16(), dp;
#pragma unroll
        for (int q4 = 0; q4 < 4; ++q4) {
            const f32x4 minus4 = *reinterpret_cast<const f32x4 *>(minus + qt * 32 + 8 * q4 + 4 * g);
#pragma unroll
            for (int e = 0; e < 4; ++e)
                dp[q4 * 4 + e] = minus4[e];
        }
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
            s = mfma(qrows.load(qt_tile, qt, ks), kf[ks], s);
            dp = mfma(qrows.load(gt_tile, qt, ks), vf[ks], dp);
        }
        // the causal mask costs three instructions per score: only in the half tiles that straddle the
        // diagonal (a wave-uniform branch; as a per-element condition it is paid everywhere)
        auto probabilities = [&](auto masked) {
#pragma unroll
            for (int q4 = 0; q4 < 4; ++q4) {
                const int at = qt * 32 + 8 * q4 + 4 * g;
                const f32x4 lse4 = *reinterpret_cast<const f32x4 *>(lse2 + at);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int r = q4 * 4 + e;
                    float p = exp2_fast(fmaf(s[r], c, -lse4[e]));
                    if (decltype(masked)::value && krow > q0 + at + e)
                        p = 0.f;
                    s[r] = p;
                    dp[r] = p * dp[r];
                }
            }
        };
        if (qh < wave_k0 + 31)
            probabilities(Const<1>{});
        else
            probabilities(Const<0>{});
#pragma unroll
        for (int kk2 = 0; kk2 < 2; ++kk2) {
            const bf16x8 pf = acc_to_frag(s, kk2);
            const bf16x8 dsf = acc_to_frag(dp, kk2);
#pragma unroll
            for (int dt = 0; dt < 2; ++dt) {
                dv[dt] = mfma(qcols.load(gt_tile, qt * 2 + kk2, dt), pf, dv[dt]);
                dk[dt] = mfma(qcols.load(qt_tile, qt * 2 + kk2, dt), dsf, dk[dt]);
            }
        }
    };
    half(Const<0>{});
    half(Const<1>{});
}
// the row's dot product with the fragments of another
TG_DEVICE float row_product(const bf16x8 (&f)[4], const bf16_t *row, int g) {
    float sum = 0.f;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
        const bf16x8 of = *reinterpret_cast<const bf16x8 *>(row + g * 8 + ks * 16);
#pragma unroll
        for (int e = 0; e < 8; ++e)
            sum += float(f[ks][e]) * float(of[e]);
    }
    return halves_sum(sum);
}
// row fragments of 32 rows: row lane % 32, 8 of every 16 columns
TG_DEVICE void load_row_fragments(bf16x8 (&f)[4], const bf16_t *row, int g) {
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
        f[ks] = *reinterpret_cast<const bf16x8 *>(row + g * 8 + ks * 16);
}

// ---------------------------------------------------------------------------------------------
// forward: block = 128 queries (4 waves x 32), key/value tiles of 64 in three LDS stages filled by
// asynchronous copies issued two tiles ahead; heavy (late) query tiles first.  The tile loop is
// unrolled by the stage count so every LDS address is a per-lane constant plus an immediate; three
// resident waves per SIMD overlap one wave's softmax with another's matrix work.
// ---------------------------------------------------------------------------------------------
__global__ __launch_bounds__(256, 3) void attn_fwd_kernel(const bf16_t *__restrict__ Q,
                                                          const bf16_t *__restrict__ K,
                                                          const bf16_t *__restrict__ V, int ld,
                                                          bf16_t *__restrict__ O, int ldo,
                                                          float *__restrict__ LSE, int T, CausalGrid grid, float c) {
    __shared__ __align__(1024) bf16_t stages[3][2][TILE_ELEMS]; // [stage][K | V]
    const CausalBlock block = grid.block(blockIdx.x);
    if (!block.live)
        return;
    const int q0 = (T / 128 - 1 - block.rank) * 128, h = block.h, b = block.b;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, g = lane >> 5;
    const int wave_q0 = q0 + wave * 32, qrow = wave_q0 + (lane & 31);
    const size_t token0 = size_t(b) * T;
    const int tiles = (q0 + 128) / 64;
    const int my_tiles = wave_q0 / 64 + 1; // tiles with a key visible to this wave (wave uniform)
    const bf16_t *kbase = K + token0 * ld + h * HD, *vbase = V + token0 * ld + h * HD;
    const uint32_t lds0 = lds_address(&stages[0][0][0]);
    // a copy takes a wave-uniform tile address and a per-lane byte offset computed once: no vector arithmetic per tile
    const uint32_t lane_offset[2] = {tile_copy_offset(ld, wave, lane, 0), tile_copy_offset(ld, wave, lane, 1)};
    auto produce = [&](int stage, int j) {
        const uint32_t slot = lds0 + uint32_t(stage) * (2 * TILE_ELEMS * 2);
        const bf16_t *kt = kbase + size_t(j) * 64 * ld, *vt = vbase + size_t(j) * 64 * ld;
#pragma unroll
        for (int n = 0; n < 2; ++n) {
            async_copy16(__builtin_amdgcn_readfirstlane(slot + (wave + 4 * n) * 1024), kt, lane_offset[n]);
            async_copy16(__builtin_amdgcn_readfirstlane(slot + TILE_ELEMS * 2 + (wave + 4 * n) * 1024), vt, lane_offset[n]);
        }
    };
    produce(0, 0);
    if (tiles > 1)
        produce(1, 1);

    bf16x8 qf[4];
    load_row_fragments(qf, Q + (token0 + qrow) * ld + h * HD, g);
    f32x16 o[2] = {zero16(), zero16()};
    float m = -INFINITY, l = 0.f;
    const RowFragOffsets krows(lane);
    const ColFragOffsets vcols(lane);

    auto step = [&](auto stage_tag, int j) {
        constexpr int STAGE = decltype(stage_tag)::value;
        // tile j was issued two steps ago; only tile j+1's four copies may still be in flight
        if (j + 1 < tiles)
            wait_vmcnt<4>();
        else
            wait_vmcnt<0>();
        __syncthreads(); // tile j visible to every wave; everyone is done with tile j-1's stage
        // the copies of tile j+2 go out at the end of the step, where the waves have drifted apart: behind
        // the barrier every wave of the CU would queue its copies at the same moment
        if (j >= my_tiles) {
            if (j + 2 < tiles)
                produce((STAGE + 2) % 3, j + 2);
            return;
        }
        f32x16 s[2];
        scores(stages[STAGE][0], krows, qf, s);
        const float before = m, alpha = online_softmax<false>(s, j * 64, wave_q0, qrow, g, c, m, l);
        if (__builtin_amdgcn_ballot_w64(m != before)) { // rescale only when some row's maximum moved
#pragma unroll
            for (int dt = 0; dt < 2; ++dt)
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    o[dt][r] *= alpha;
        }
        weigh_values(stages[STAGE][1], vcols, s, o);
        if (j + 2 < tiles)
            produce((STAGE + 2) % 3, j + 2);
    };
    for (int j = 0; j < tiles; j += 3) { // tiles is block uniform
        step(Const<0>{}, j);
        if (j + 1 < tiles)
            step(Const<1>{}, j + 1);
        if (j + 2 < tiles)
            step(Const<2>{}, j + 2);
    }
    l = halves_sum(l);
    const float inv = 1.0f / l;
    bf16_t *op = O + (token0 + qrow) * ldo + h * HD;
#pragma unroll
    for (int dt = 0; dt < 2; ++dt)
        store_acc_rows(op + dt * 32, o[dt], inv, g);
    if (g == 0)
        LSE[(size_t(b) * grid.H + h) * T + qrow] = (m + __log2f(l)) * LN2;
}

// ---------------------------------------------------------------------------------------------
// dK, dV: block = 128 keys (4 waves x 32), loops over 64-query tiles from the diagonal on; Q and dO
// tiles (plus the 64 log-sum-exps and deltas of the tile) arrive by asynchronous copies two tiles
// ahead.  Scores are produced as S[query][key] here: one lane owns one KEY, which is the row index
// of both outputs.  The two 32-query halves of a tile are processed one after the other to keep the
// live accumulators, and with them the register count, down.
// ---------------------------------------------------------------------------------------------
typedef bf16_t TileStages[3][2][TILE_ELEMS];
typedef float RowStages[3][2][64];
TG_DEVICE void dkdv_block(TileStages &stages /* [stage][Q | dO] */, RowStages &rows /* [stage][lse2 | -delta] */,
                          const CausalBlock &block, const CausalGrid &grid, const bf16_t *__restrict__ Q,
                          const bf16_t *__restrict__ K, const bf16_t *__restrict__ V, int ld, const bf16_t *__restrict__ dO,
                          int lddo, const float *__restrict__ lse2, const float *__restrict__ delta, bf16_t *__restrict__ dK,
                          bf16_t *__restrict__ dV, int lddq, int T, float scale) {
    const int k0 = block.rank * 128, h = block.h, b = block.b; // early keys see the most queries
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, g = lane >> 5;
    const int wave_k0 = k0 + wave * 32, krow = wave_k0 + (lane & 31);
    const size_t token0 = size_t(b) * T;
    const float c = scale * LOG2E;
    const int first = k0 / 64, tiles = T / 64 - first;
    const bf16_t *qbase = Q + (token0 + first * 64) * ld + h * HD;
    const bf16_t *gbase = dO + (token0 + first * 64) * lddo + h * HD;
    const float *row_source = ((wave & 1) ? delta : lse2) + (size_t(b) * grid.H + h) * T + first * 64 + lane;
    const uint32_t lds0 = lds_address(&stages[0][0][0]), rows0 = lds_address(&rows[0][wave & 1][0]);
    const uint32_t q_offset[2] = {tile_copy_offset(ld, wave, lane, 0), tile_copy_offset(ld, wave, lane, 1)};
    const uint32_t g_offset[2] = {tile_copy_offset(lddo, wave, lane, 0), tile_copy_offset(lddo, wave, lane, 1)};
    auto produce_one = [&](int stage, int j, int n) { // n-th of a wave's five copies for tile j
        const uint32_t slot = lds0 + uint32_t(stage) * (2 * TILE_ELEMS * 2);
        if (n < 2)
            async_copy16(__builtin_amdgcn_readfirstlane(slot + (wave + 4 * n) * 1024), qbase + size_t(j) * 64 * ld,
                         q_offset[n]);
        else if (n < 4)
            async_copy16(__builtin_amdgcn_readfirstlane(slot + TILE_ELEMS * 2 + (wave + 4 * (n - 2)) * 1024),
                         gbase + size_t(j) * 64 * lddo, g_offset[n - 2]);
        else
            async_copy4(__builtin_amdgcn_readfirstlane(rows0 + uint32_t(stage) * (2 * 64 * 4)), row_source + j * 64);
    };
    auto produce = [&](int stage, int j) {
#pragma unroll
        for (int n = 0; n < 5; ++n)
            produce_one(stage, j, n);
    };
    produce(0, 0);
    produce(1, tiles > 1 ? 1 : 0);

    bf16x8 kf[4], vf[4];
    load_row_fragments(kf, K + (token0 + krow) * ld + h * HD, g);
    load_row_fragments(vf, V + (token0 + krow) * ld + h * HD, g);
    f32x16 dk[2] = {zero16(), zero16()}, dv[2] = {zero16(), zero16()};
    const RowFragOffsets qrows(lane);
    const ColFragOffsets qcols(lane);

    auto step = [&](auto stage_tag, int j) {
        constexpr int STAGE = decltype(stage_tag)::value;
        wait_vmcnt<5>(); // only the five copies issued during tile j-1 may still be in flight
        __syncthreads(); // tile j visible to every wave; everyone is done with tile j-1's stage
        // The copies of tile j+2 go out at the end of the step, where the waves have drifted apart: behind the
        // barrier all eight waves of the CU queue theirs at once and wait for one another (measured -2 %).
        // Every step issues five (past the end the last tile once more, into the stage nobody reads any
        // more), so the wait above is always the same.
        const int ahead = j + 2 < tiles ? j + 2 : tiles - 1;
        dkdv_tile(stages[STAGE][0], stages[STAGE][1], rows[STAGE][0], rows[STAGE][1], (first + j) * 64, wave_k0, krow, g, c,
                  qrows, qcols, kf, vf, dk, dv);
        produce((STAGE + 2) % 3, ahead);
    };
    for (int j = 0; j < tiles; j += 3) { // tiles is block uniform
        step(Const<0>{}, j);
        if (j + 1 < tiles)
            step(Const<1>{}, j + 1);
        if (j + 2 < tiles)
            step(Const<2>{}, j + 2);
    }
    wait_vmcnt<0>(); // no copy may land in LDS after the block has left
    bf16_t *kp = dK + (token0 + krow) * lddq + h * HD;
    bf16_t *vp = dV + (token0 + krow) * lddq + h * HD;
#pragma unroll
    for (int dt = 0; dt < 2; ++dt) {
        store_acc_rows(kp + dt * 32, dk[dt], scale, g);
        store_acc_rows(vp + dt * 32, dv[dt], 1.0f, g);
    }
}

__global__ __launch_bounds__(256, 2) void attn_bwd_dkdv_kernel(
    const bf16_t *__restrict__ Q, const bf16_t *__restrict__ K, const bf16_t *__restrict__ V, int ld,
    const bf16_t *__restrict__ dO, int lddo, const float *__restrict__ lse2,
    const float *__restrict__ delta, bf16_t *__restrict__ dK, bf16_t *__restrict__ dV, int lddq, int T, CausalGrid grid, float scale) {
    __shared__ __align__(1024) TileStages stages;
    __shared__ __align__(256) RowStages rows;
    const CausalBlock block = grid.block(blockIdx.x);
    if (block.live)
        dkdv_block(stages, rows, block, grid, Q, K, V, ld, dO, lddo, lse2, delta, dK, dV, lddq, T, scale);
}

// ---------------------------------------------------------------------------------------------
// dQ: block = 128 queries (4 waves x 32), loops over 64-key tiles up to the diagonal; K and V tiles
// arrive by asynchronous copies two tiles ahead; 32-key halves are processed in turn.
// ---------------------------------------------------------------------------------------------
// `lse2_out` and `delta_out` may be NULL.
TG_DEVICE void dq_block(TileStages &stages /* [stage][K | V] */, const CausalBlock &block, const CausalGrid &grid,
                        const bf16_t *__restrict__ Q, const bf16_t *__restrict__ K, const bf16_t *__restrict__ V, int ld,
                        const bf16_t *__restrict__ dO, int lddo, const bf16_t *__restrict__ O, int ldo,
                        const float *__restrict__ LSE, float *__restrict__ lse2_out, float *__restrict__ delta_out,
                        bf16_t *__restrict__ dQ, int lddq, int T, float scale) {
    const int q0 = (T / 128 - 1 - block.rank) * 128, h = block.h, b = block.b;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, g = lane >> 5;
    const int wave_q0 = q0 + wave * 32, qrow = wave_q0 + (lane & 31);
    const size_t token0 = size_t(b) * T;
    const float c = scale * LOG2E;
    const int tiles = (q0 + 128) / 64;
    const int my_tiles = wave_q0 / 64 + 1;
    const bf16_t *kbase = K + token0 * ld + h * HD, *vbase = V + token0 * ld + h * HD;
    const uint32_t lds0 = lds_address(&stages[0][0][0]);
    // a copy takes a wave-uniform tile address and a per-lane byte offset computed once: no vector arithmetic per tile
    const uint32_t lane_offset[2] = {tile_copy_offset(ld, wave, lane, 0), tile_copy_offset(ld, wave, lane, 1)};
    auto produce = [&](int stage, int j) {
        const uint32_t slot = lds0 + uint32_t(stage) * (2 * TILE_ELEMS * 2);
        const bf16_t *kt = kbase + size_t(j) * 64 * ld, *vt = vbase + size_t(j) * 64 * ld;
#pragma unroll
        for (int n = 0; n < 2; ++n) {
            async_copy16(__builtin_amdgcn_readfirstlane(slot + (wave + 4 * n) * 1024), kt, lane_offset[n]);
            async_copy16(__builtin_amdgcn_readfirstlane(slot + TILE_ELEMS * 2 + (wave + 4 * n) * 1024), vt, lane_offset[n]);
        }
    };
    produce(0, 0);
    if (tiles > 1)
        produce(1, 1);

    bf16x8 qf[4], gf[4];
    load_row_fragments(qf, Q + (token0 + qrow) * ld + h * HD, g);
    load_row_fragments(gf, dO + (token0 + qrow) * lddo + h * HD, g);
    // delta = rowsum(dO o O) and the log-sum-exp in base 2, for this block's own queries; also left in
    // memory for the dK/dV kernel, which runs after this one
    const float del = row_product(gf, O + (token0 + qrow) * ldo + h * HD, g);
    const size_t row_at = (size_t(b) * grid.H + h) * T + qrow;
    const float lse = LSE[row_at] * LOG2E;
    if (g == 0 && delta_out) {
        delta_out[row_at] = -del; // negated: the dK/dV kernel starts its dP product from it
        lse2_out[row_at] = lse;
    }
    f32x16 dq[2] = {zero16(), zero16()};
    f32x16 minus_delta;
#pragma unroll
    for (int r = 0; r < 16; ++r)
        minus_delta[r] = -del;
    const RowFragOffsets krows(lane);
    const ColFragOffsets kcols(lane);

    auto step = [&](auto stage_tag, int j) {
        constexpr int STAGE = decltype(stage_tag)::value;
        if (j + 1 < tiles)
            wait_vmcnt<4>();
        else
            wait_vmcnt<0>();
        __syncthreads();
        // the copies of tile j+2 go out at the end of the step, where the waves have drifted apart: behind
        // the barrier every wave of the CU would queue its copies at the same moment
        if (j >= my_tiles) {
            if (j + 2 < tiles)
                produce((STAGE + 2) % 3, j + 2);
            return;
        }
        dq_tile(stages[STAGE][0], stages[STAGE][1], j * 64, wave_q0, qrow, g, c, lse, krows, kcols, qf, gf, minus_delta, dq);
        if (j + 2 < tiles)
            produce((STAGE + 2) % 3, j + 2);
    };
    for (int j = 0; j < tiles; j += 3) { // tiles is block uniform
        step(Const<0>{}, j);
        if (j + 1 < tiles)
            step(Const<1>{}, j + 1);
        if (j + 2 < tiles)
            step(Const<2>{}, j + 2);
    }
    bf16_t *qp = dQ + (token0 + qrow) * lddq + h * HD;
#pragma unroll
    for (int dt = 0; dt < 2; ++dt)
        store_acc_rows(qp + dt * 32, dq[dt], scale, g);
}

__global__ __launch_bounds__(256, 3) void attn_bwd_dq_kernel(
    const bf16_t *__restrict__ Q, const bf16_t *__restrict__ K, const bf16_t *__restrict__ V, int ld,
    const bf16_t *__restrict__ dO, int lddo, const bf16_t *__restrict__ O, int ldo,
    const float *__restrict__ LSE, float *__restrict__ lse2_out, float *__restrict__ delta_out,
    bf16_t *__restrict__ dQ, int lddq, int T, CausalGrid grid, float scale) {
    __shared__ __align__(1024) TileStages stages;
    const CausalBlock block = grid.block(blockIdx.x);
    if (block.live)
        dq_block(stages, block, grid, Q, K, V, ld, dO, lddo, O, ldo, LSE, lse2_out, delta_out, dQ, lddq, T, scale);
}

// ---------------------------------------------------------------------------------------------
// The two side by side, where neither fills the units (backward_way has the rule): every other run of eight blocks takes
// 128 keys, the others 128 queries, and a launch before them leaves the deltas, which the dQ kernel otherwise hands on.
// ---------------------------------------------------------------------------------------------
__global__ __launch_bounds__(256, 2) void attn_bwd_both_kernel(
    const bf16_t *__restrict__ Q, const bf16_t *__restrict__ K, const bf16_t *__restrict__ V, int ld,
    const bf16_t *__restrict__ dO, int lddo, const bf16_t *__restrict__ O, int ldo, const float *__restrict__ LSE,
    const float *__restrict__ lse2, const float *__restrict__ delta, bf16_t *__restrict__ dQ, bf16_t *__restrict__ dK,
    bf16_t *__restrict__ dV, int lddq, int T, CausalGrid grid, float scale) {
    __shared__ __align__(1024) TileStages stages;
    __shared__ __align__(256) RowStages rows;
    const CausalBlock block = grid.block((blockIdx.x >> 4) * 8 + (blockIdx.x & 7));
    if (!block.live)
        return;
    if (blockIdx.x & 8)
        dq_block(stages, block, grid, Q, K, V, ld, dO, lddo, O, ldo, LSE, nullptr, nullptr, dQ, lddq, T, scale);
    else
        dkdv_block(stages, rows, block, grid, Q, K, V, ld, dO, lddo, lse2, delta, dK, dV, lddq, T, scale);
}
// -rowsum(dO o O) and the log-sum-exp in base 2 of every row: eight lanes a row, eight consecutive queries a wave
__global__ __launch_bounds__(256) void attn_delta_kernel(const bf16_t *__restrict__ dO, int lddo, const bf16_t *__restrict__ O,
                                                         int ldo, const float *__restrict__ LSE, float *__restrict__ lse2,
                                                         float *__restrict__ delta, int H, int T) {
    const int per_head = T / 32, head = blockIdx.x / per_head, t = (blockIdx.x - head * per_head) * 32 + (threadIdx.x >> 3);
    const int b = head / H, h = head - b * H, part = threadIdx.x & 7;
    const size_t token = size_t(b) * T + t, row = size_t(head) * T + t;
    const u32x4 x = *reinterpret_cast<const u32x4 *>(dO + token * lddo + h * HD + part * 8);
    const u32x4 y = *reinterpret_cast<const u32x4 *>(O + token * ldo + h * HD + part * 8);
    float sum = 0.f;
#pragma unroll
    for (int e = 0; e < 4; ++e)
        sum = fmaf(bf16_hi(x[e]), bf16_hi(y[e]), fmaf(bf16_lo(x[e]), bf16_lo(y[e]), sum));
#pragma unroll
    for (int k = 1; k < 8; k <<= 1)
        sum += __shfl_xor(sum, k, 64);
    if (part == 0) {
        delta[row] = -sum;
        lse2[row] = LSE[row] * LOG2E;
    }
}

// ---------------------------------------------------------------------------------------------
// Few rows.  A wave of the kernels above walks its row's tiles one after another, T/64 of them at worst, at about
// 0.8 us each, whatever the number of blocks: with one block of 128 rows per compute unit or less that chain is the
// kernel's time and most SIMDs are idle or wait.  Here a block is 32 queries (or keys) and its four waves take the
// tiles of the other side in turn, each into a stage of its own (no barrier in the loop) and with sums of its own,
// which meet in LDS at the end: a chain a quarter as long on four times the blocks.  The price is that a tile is
// fetched once per 32 rows instead of once per 128 and that the stages are not double buffered (two blocks of 64 KiB
// per compute unit fill in for each other); the backward is one launch, because its dK/dV blocks form the deltas of
// their queries themselves.  Microseconds, 128-row blocks -> these (B, H, T), forward; backward:
//   1,1,128: 4.6 -> 4.0; 11.6 -> 4.9    8,4,256: 6.5 -> 4.7; 16.7 -> 7.5
//   1,12,1024: 16.1 -> 8.1; 42.1 -> 17.2    1,4,4096: 53 -> 20; 144 -> 51    1,1,8192: 99 -> 29; 273 -> 68
// What bounds the short ones is the copy path: of the backward's 8.2 us at 8,4,256 (back to back in a graph, where an empty launch
// takes 1.6) loads and joins alone were 6.1.  The fragments of the block's own 32 rows were a quarter line a lane and load, in
// each of four waves, and so was O for the deltas.  The own rows now come to LDS once, O as whole lines, and a lane multiplies what
// it holds of a row: 8,4,256 8.2 -> 6.6, 1,16,1024 26.0 -> 21.1, 1,2,8192 103 -> 94; forward 4.4 -> 4.2, 8.2 -> 7.8, 37.4 -> 34.7.
// ---------------------------------------------------------------------------------------------
constexpr int WAVES = 4;
// this wave's own 64 x 64 tile, rows ld elements apart, in eight copies
struct WaveTileCopy {
    uint32_t offset[2];
    int ld;
    TG_DEVICE WaveTileCopy(int ld_, int lane) : offset{tile_copy_offset(ld_, 0, lane, 0), tile_copy_offset(ld_, 1, lane, 0)}, ld(ld_) {}
    TG_DEVICE void operator()(uint32_t lds_tile, const bf16_t *base) const {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int odd = 0; odd < 2; ++odd)
                async_copy16(__builtin_amdgcn_readfirstlane(lds_tile + (2 * i + odd) * 1024), base + size_t(i) * 16 * ld, offset[odd]);
    }
};
// The block's own 32 rows, the first half of a tile's image, eight to a wave.  Read from there they are four fragments a wave for
// one copy; as fragments from memory each of the four waves asks for 32 lines of which it takes a quarter at a time.
TG_DEVICE void copy_own_rows(bf16_t *half_tile, const bf16_t *base, int ld, int wave, int lane) {
    async_copy16(__builtin_amdgcn_readfirstlane(lds_address(half_tile) + wave * 1024), base, tile_copy_offset(ld, wave, lane, 0));
}
TG_DEVICE void own_fragments(bf16x8 (&f)[4], const bf16_t *half_tile, const RowFragOffsets &along) {
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
        f[ks] = along.load(half_tile, 0, ks);
}
// Rows' dot products, a row to eight lanes.  First this lane's part: of what it copied to `copied` with the same 16 bytes of another
// matrix.  Lane 4 b + i holds row i of both factors of block b of the 4 x 4 x 4 instruction, so its part stands on the diagonal: two
// such instructions and three selections where unpacking and multiplying takes 25 vector instructions.
TG_DEVICE float chunk_product(const unsigned char *copied, const u32x4 &other, int lane) {
    const u32x4 mine = *reinterpret_cast<const u32x4 *>(copied);
    const auto four = [](uint32_t x, uint32_t y) { return __builtin_bit_cast(s16x4, u32x2{x, y}); };
    f32x4 sum = {0.f, 0.f, 0.f, 0.f};
    sum = __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(four(mine[0], mine[1]), four(other[0], other[1]), sum, 0, 0, 0);
    sum = __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(four(mine[2], mine[3]), four(other[2], other[3]), sum, 0, 0, 0);
    const float even = lane & 2 ? sum[2] : sum[0], odd = lane & 2 ? sum[3] : sum[1];
    return lane & 1 ? odd : even;
}
// the value of another of the eight lanes: the neighbour, the one two further on, the one opposite
constexpr int NEIGHBOUR = 0xB1, TWO_ON = 0x4E, OPPOSITE = 0x141;
template <int WHICH> TG_DEVICE float from_lane(float x) {
    return __uint_as_float(uint32_t(__builtin_amdgcn_update_dpp(0, int(__float_as_uint(x)), WHICH, 0xF, 0xF, true)));
}
TG_DEVICE float eight_lanes_sum(float x) {
    x += from_lane<OPPOSITE>(x);
    x += from_lane<TWO_ON>(x);
    return x + from_lane<NEIGHBOUR>(x);
}
// part[i] summed over the eight lanes, in the lane with lane % 8 = i: each step keeps the half that the lane is in
TG_DEVICE float eight_sums(const float (&part)[8], int lane) {
    float four[4], two[2];
#pragma unroll
    for (int i = 0; i < 4; ++i)
        four[i] = (lane & 4 ? part[i + 4] : part[i]) + from_lane<OPPOSITE>(lane & 4 ? part[i] : part[i + 4]);
#pragma unroll
    for (int i = 0; i < 2; ++i)
        two[i] = (lane & 2 ? four[i + 2] : four[i]) + from_lane<TWO_ON>(lane & 2 ? four[i] : four[i + 2]);
    return (lane & 1 ? two[1] : two[0]) + from_lane<NEIGHBOUR>(lane & 1 ? two[0] : two[1]);
}
// a wave's 32 x 64 sums to its part of LDS, 16 bytes a lane and store
TG_DEVICE void leave_sums(float *part, const f32x16 (&acc)[2], int lane) {
#pragma unroll
    for (int n = 0; n < 8; ++n)
        *reinterpret_cast<f32x4 *>(part + (n * 64 + lane) * 4) =
            f32x4{acc[n >> 2][(n & 3) * 4], acc[n >> 2][(n & 3) * 4 + 1], acc[n >> 2][(n & 3) * 4 + 2], acc[n >> 2][(n & 3) * 4 + 3]};
}
// columns 16 * wave .. +15 of the block's 32 rows: eight sums a lane, of the `parts` waves that had a tile
TG_DEVICE void join_sums(float (&sum)[8], const float *part0, size_t stride, int parts, const float *weight, int wave, int lane) {
#pragma unroll
    for (int e = 0; e < 8; ++e)
        sum[e] = 0.f;
#pragma unroll
    for (int w = 0; w < WAVES; ++w)
        if (w < parts) {
            const float *from = part0 + w * stride + (wave * 2 * 64 + lane) * 4;
            const f32x4 lo = *reinterpret_cast<const f32x4 *>(from), hi = *reinterpret_cast<const f32x4 *>(from + 256);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                sum[e] = fmaf(lo[e], weight[w], sum[e]);
                sum[e + 4] = fmaf(hi[e], weight[w], sum[e + 4]);
            }
        }
}
TG_DEVICE void store_joined(bf16_t *row, const float (&sum)[8], float scale, int wave, int g) {
    const auto x = __builtin_amdgcn_permlane32_swap(pack_bf16(sum[0] * scale, sum[1] * scale),
                                                    pack_bf16(sum[4] * scale, sum[5] * scale), false, false);
    const auto y = __builtin_amdgcn_permlane32_swap(pack_bf16(sum[2] * scale, sum[3] * scale),
                                                    pack_bf16(sum[6] * scale, sum[7] * scale), false, false);
    *reinterpret_cast<u32x4 *>(row + wave * 16 + 8 * g) = u32x4{x[0], y[0], x[1], y[1]};
}

// SHARED: the queries come by way of LDS.  At 128 positions only one or two waves want them, which have them sooner from memory.
template <bool SHARED>
__global__ __launch_bounds__(256, 2) void attn_fwd_split_kernel(const bf16_t *__restrict__ Q, const bf16_t *__restrict__ K,
                                                                const bf16_t *__restrict__ V, int ld, bf16_t *__restrict__ O,
                                                                int ldo, float *__restrict__ LSE, int T, CausalGrid grid, float c) {
    __shared__ __align__(1024) bf16_t tile[WAVES][2][TILE_ELEMS]; // [wave][K | V], then the waves' sums
    __shared__ float2 row_sums[WAVES][32];                        // maximum and sum of a row
    const CausalBlock block = grid.block(blockIdx.x);
    if (!block.live)
        return;
    const int q0 = (T / 32 - 1 - block.rank) * 32, h = block.h, b = block.b;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), g = lane >> 5, qrow = q0 + (lane & 31);
    const size_t token0 = size_t(b) * T;
    const int tiles = q0 / 64 + 1;
    const bf16_t *kbase = K + token0 * ld + h * HD, *vbase = V + token0 * ld + h * HD;
    const uint32_t slot = lds_address(&tile[wave][0][0]);
    const WaveTileCopy copy(ld, lane);
    bf16x8 qf[4];
    f32x16 o[2] = {zero16(), zero16()};
    float m = -INFINITY, l = 0.f;
    const RowFragOffsets krows(lane);
    const auto first_tile = [&] {
        copy(slot, kbase + size_t(wave) * 64 * ld);
        copy(slot + TILE_ELEMS * 2, vbase + size_t(wave) * 64 * ld);
    };
    if constexpr (SHARED) {
        __shared__ __align__(1024) bf16_t own[TILE_ELEMS / 2];
        copy_own_rows(own, Q + (token0 + q0) * ld + h * HD, ld, wave, lane);
        if (wave < tiles) {
            first_tile();
            wait_vmcnt<8>(); // the queries and the first tile's keys are there, its values may still be on the way
        } else {
            wait_vmcnt<0>();
        }
        __syncthreads();
        own_fragments(qf, own, krows);
    } else if (wave < tiles) {
        first_tile();
        load_row_fragments(qf, Q + (token0 + qrow) * ld + h * HD, g);
    }
    if (wave < tiles) {
        const ColFragOffsets vcols(lane);
        for (int j = wave; j < tiles; j += WAVES) {
            const bool more = j + WAVES < tiles;
            f32x16 s[2];
            wait_vmcnt<8>(); // this tile's keys are there, its values may still be on the way
            scores(tile[wave][0], krows, qf, s);
            if (more) {
                wait_lgkmcnt0(); // the keys have been read
                copy(slot, kbase + size_t(j + WAVES) * 64 * ld);
            }
            const float before = m, alpha = online_softmax<true>(s, j * 64, q0, qrow, g, c, m, l);
            if (__builtin_amdgcn_ballot_w64(m != before)) {
#pragma unroll
                for (int dt = 0; dt < 2; ++dt)
#pragma unroll
                    for (int r = 0; r < 16; ++r)
                        o[dt][r] *= alpha;
            }
            if (more)
                wait_vmcnt<8>();
            else
                wait_vmcnt<0>();
            weigh_values(tile[wave][1], vcols, s, o);
            if (more) {
                wait_lgkmcnt0();
                copy(slot + TILE_ELEMS * 2, vbase + size_t(j + WAVES) * 64 * ld);
            }
        }
        wait_lgkmcnt0(); // the tile has been read
        l = halves_sum(l);
        leave_sums(reinterpret_cast<float *>(tile[wave]), o, lane);
        if (g == 0)
            row_sums[wave][lane] = make_float2(m, l);
    }
    __syncthreads();
    const int parts = tiles < WAVES ? tiles : WAVES;
    float weight[WAVES], top = -INFINITY, total = 0.f, sum[8];
#pragma unroll
    for (int w = 0; w < WAVES; ++w)
        if (w < parts)
            top = fmaxf(top, row_sums[w][lane & 31].x);
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
        weight[w] = 0.f;
        if (w < parts) {
            const float2 row = row_sums[w][lane & 31];
            weight[w] = exp2_fast(row.x - top);
            total = fmaf(row.y, weight[w], total);
        }
    }
    join_sums(sum, reinterpret_cast<const float *>(tile[0]), sizeof(tile[0]) / sizeof(float), parts, weight, wave, lane);
    store_joined(O + (token0 + qrow) * ldo + h * HD, sum, 1.0f / total, wave, g);
    if (threadIdx.x < 32)
        LSE[(size_t(b) * grid.H + h) * T + qrow] = (top + __log2f(total)) * LN2;
}

// dK, dV and dQ in one launch: every other run of eight blocks takes 32 keys, the others 32 queries
__global__ __launch_bounds__(256, 2) void attn_bwd_split_kernel(
    const bf16_t *__restrict__ Q, const bf16_t *__restrict__ K, const bf16_t *__restrict__ V, int ld,
    const bf16_t *__restrict__ dO, int lddo, const bf16_t *__restrict__ O, int ldo, const float *__restrict__ LSE,
    bf16_t *__restrict__ dQ, bf16_t *__restrict__ dK, bf16_t *__restrict__ dV, int lddq, int T, CausalGrid grid, float scale) {
    __shared__ __align__(1024) bf16_t tile[WAVES][2][TILE_ELEMS]; // [wave][Q | dO] or [K | V], then the waves' sums
    __shared__ __align__(1024) bf16_t own[2][TILE_ELEMS / 2];     // K | V or Q | dO
    __shared__ __align__(256) float rows[WAVES][2][64];           // [wave][lse2 | -delta]
    const CausalBlock block = grid.block((blockIdx.x >> 4) * 8 + (blockIdx.x & 7));
    if (!block.live)
        return;
    const bool keys = !(blockIdx.x & 8);
    const int h = block.h, b = block.b;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), g = lane >> 5;
    const size_t token0 = size_t(b) * T;
    const float c = scale * LOG2E;
    const float *lse_row = LSE + (size_t(b) * grid.H + h) * T;
    const uint32_t slot = lds_address(&tile[wave][0][0]);
    float *part = reinterpret_cast<float *>(tile[wave]);
    const float *part0 = reinterpret_cast<const float *>(tile[0]);
    constexpr size_t STRIDE = sizeof(tile[0]) / sizeof(float);
    const float ones[WAVES] = {1.f, 1.f, 1.f, 1.f};
    float sum[8];
    const RowFragOffsets along(lane);
    const ColFragOffsets across(lane);
    if (keys) {
        const int k0 = block.rank * 32, krow = k0 + (lane & 31), first = k0 / 64, tiles = T / 64 - first;
        copy_own_rows(own[0], K + (token0 + k0) * ld + h * HD, ld, wave, lane);
        copy_own_rows(own[1], V + (token0 + k0) * ld + h * HD, ld, wave, lane);
        const WaveTileCopy copy_q(ld, lane), copy_g(lddo, lane);
        const uint32_t o_offset[2] = {tile_copy_offset(ldo, 0, lane, 0), tile_copy_offset(ldo, 1, lane, 0)};
        u32x4 of[8];
        float lse = 0.f;
        // a tile's copies to LDS, and its O as the copies of dO lie
        const auto request = [&](int q0) {
            copy_q(slot, Q + (token0 + q0) * ld + h * HD);
            copy_g(slot + TILE_ELEMS * 2, dO + (token0 + q0) * lddo + h * HD);
            const char *o = reinterpret_cast<const char *>(O + (token0 + q0) * ldo + h * HD);
#pragma unroll
            for (int i = 0; i < 8; ++i)
                of[i] = *reinterpret_cast<const u32x4 *>(o + size_t(i >> 1) * 32 * ldo + o_offset[i & 1]);
            lse = lse_row[q0 + lane];
        };
        if (wave < tiles)
            request((first + wave) * 64);
        wait_vmcnt<0>();
        __syncthreads();
        if (wave < tiles) {
            bf16x8 kf[4], vf[4];
            own_fragments(kf, own[0], along);
            own_fragments(vf, own[1], along);
            f32x16 dk[2] = {zero16(), zero16()}, dv[2] = {zero16(), zero16()};
            for (int j = wave; j < tiles; j += WAVES) {
                const int q0 = (first + j) * 64;
                if (j != wave) {
                    request(q0);
                    wait_vmcnt<0>();
                }
                rows[wave][0][lane] = lse * LOG2E;
                // deltas of the tile's queries: this lane gets that of row 8 * (lane % 8) + lane / 8
                float part[8];
#pragma unroll
                for (int i = 0; i < 8; ++i)
                    part[i] = chunk_product(reinterpret_cast<const unsigned char *>(tile[wave][1]) + i * 1024 + lane * 16, of[i], lane);
                rows[wave][1][(lane & 7) * 8 + (lane >> 3)] = -eight_sums(part, lane);
                dkdv_tile(tile[wave][0], tile[wave][1], rows[wave][0], rows[wave][1], q0, k0, krow, g, c, along, across, kf, vf,
                          dk, dv);
                wait_lgkmcnt0(); // the tile has been read
            }
            leave_sums(part, dk, lane);
            leave_sums(part + TILE_ELEMS / 2, dv, lane);
        }
        __syncthreads();
        const int parts = tiles < WAVES ? tiles : WAVES;
        join_sums(sum, part0, STRIDE, parts, ones, wave, lane);
        store_joined(dK + (token0 + krow) * lddq + h * HD, sum, scale, wave, g);
        join_sums(sum, part0 + TILE_ELEMS / 2, STRIDE, parts, ones, wave, lane);
        store_joined(dV + (token0 + krow) * lddq + h * HD, sum, 1.0f, wave, g);
    } else {
        const int q0 = (T / 32 - 1 - block.rank) * 32, qrow = q0 + (lane & 31), tiles = q0 / 64 + 1;
        const WaveTileCopy copy(ld, lane);
        const bf16_t *kbase = K + token0 * ld + h * HD, *vbase = V + token0 * ld + h * HD;
        copy_own_rows(own[0], Q + (token0 + q0) * ld + h * HD, ld, wave, lane);
        copy_own_rows(own[1], dO + (token0 + q0) * lddo + h * HD, lddo, wave, lane);
        const u32x4 of = *reinterpret_cast<const u32x4 *>(reinterpret_cast<const char *>(O + (token0 + q0) * ldo + h * HD) +
                                                          tile_copy_offset(ldo, wave, lane, 0));
        if (wave < tiles) {
            copy(slot, kbase + size_t(wave) * 64 * ld);
            copy(slot + TILE_ELEMS * 2, vbase + size_t(wave) * 64 * ld);
        }
        const float lse = lse_row[qrow] * LOG2E;
        wait_vmcnt<0>();
        const float product = eight_lanes_sum(chunk_product(reinterpret_cast<const unsigned char *>(own[1]) + wave * 1024 + lane * 16, of, lane));
        if (!(lane & 7))
            rows[0][1][wave * 8 + (lane >> 3)] = -product;
        __syncthreads();
        if (wave < tiles) {
            bf16x8 qf[4], gf[4];
            own_fragments(qf, own[0], along);
            own_fragments(gf, own[1], along);
            const float minus = rows[0][1][lane & 31];
            f32x16 dq[2] = {zero16(), zero16()};
            f32x16 minus_delta;
#pragma unroll
            for (int r = 0; r < 16; ++r)
                minus_delta[r] = minus;
            for (int j = wave; j < tiles; j += WAVES) {
                wait_vmcnt<0>();
                dq_tile(tile[wave][0], tile[wave][1], j * 64, q0, qrow, g, c, lse, along, across, qf, gf, minus_delta, dq);
                wait_lgkmcnt0();
                if (j + WAVES < tiles) {
                    copy(slot, kbase + size_t(j + WAVES) * 64 * ld);
                    copy(slot + TILE_ELEMS * 2, vbase + size_t(j + WAVES) * 64 * ld);
                }
            }
            leave_sums(part, dq, lane);
        }
        __syncthreads();
        join_sums(sum, part0, STRIDE, tiles < WAVES ? tiles : WAVES, ones, wave, lane);
        store_joined(dQ + (token0 + qrow) * lddq + h * HD, sum, scale, wave, g);
    }
}

// Up to how many 128-row blocks the 32-row ones with shared-out tiles are taken instead.  The longer the context, the
// longer the chains that they cut, so the line rises with it.  Forward, microseconds, 128-row / 32-row:
//   T 128: 128 blocks 4.6 / 4.6   144: 4.7 / 6.4     T 256: 128 blocks 6.2 / 5.2   144: 6.2 / 6.9
//   T 384: 144 blocks 7.7 / 7.2   162: 7.8 / 8.1     T 512: 192 blocks 9.4 / 9.0   256: 9.6 / 9.9
//   T 768: 252 blocks 12.7 / 11.5   288: 12.8 / 14.2     T 1024: 320 blocks 16.5 / 16.4   328: 16.8 / 16.9   352: 16.6 / 17.2
//   T 1152: 324 blocks 18.4 / 17.1   351: 18.6 / 18.7   360: 18.1 / 18.5     T 1536: 384 blocks 23.3 / 21.9   432: 24.3 / 24.9
//   T 2048: 384 blocks 29.4 / 27.1   448: 31.5 / 31.0     T 4096: 384 blocks 58.7 / 45.5   448: 60.5 / 53.7     T 8192: 448 blocks 121 / 102
// So the cap, right at 1536, comes too soon from 4096 on.  A tile's largest probability is 1 in a wave's own sums, where
// only a row's is in the longer chain: against 64 bits 32-row blocks are nearer by up to 0.8 % of the outputs' error (13,5,256 1.92e-3
// against 1.94e-3), of bf16 roundings both.
bool forward_splits(int B, int H, int T) {
    return size_t(B) * H * (T / 128) <= size_t(std::clamp(T / 4 + 64, 128, 384));
}
// The backward does five products where the forward does two and loses by the split kernel's fetches sooner.  Next come
// its two kernels side by side, as long as both sets of blocks are about what the units hold (two each).  Microseconds, split /
// side by side:
//   T 128: 128 blocks 10.5 / 10.9   144: 13.3 / 13.0     T 256: 128 blocks 11.9 / 13.3   144: 14.1 / 14.4   154: 15.2 / 14.7
//   T 384: 144 blocks 16.1 / 16.2   162: 17.4 / 16.8     T 512: 128 blocks 14.9 / 18.2   160: 18.7 / 19.0   192: 20.6 / 19.9
//   T 768: 144 blocks 20.8 / 23.6   192: 24.8 / 25.0     T 1024: 184 blocks 29.8 / 29.9     T 1280: 200 blocks 32.2 / 34.0   210: 35.4 / 34.4
//   T 1536: 204 blocks 38.2 / 39.6   216: 41.2 / 41.1     T 2048: 192 blocks 43.3 / 49.6   208: 50.6 / 49.7     T 4096: 192 blocks 80 / 92   224: 99 / 92
//   T 8192: 128 blocks 99 / 161   192: 144 / 174   256: 179 / 175
// and side by side / one after the other:
//   T 128: 256 blocks 13.5 / 14.4     T 256: 256 blocks 15.4 / 18.5   512: 28.3 / 24.6     T 512: 384 blocks 27.6 / 30.0   576: 41.5 / 37.6
//   T 1024: 512 blocks 48.9 / 50.8   768: 70.5 / 67.5     T 2048: 512 blocks 78.9 / 87.5   768: 112 / 108     T 4096: 512 blocks 141 / 163
enum Backward { BACKWARD_SPLIT, BACKWARD_BOTH, BACKWARD_IN_TURN };
Backward backward_way(int B, int H, int T) {
    const size_t blocks = size_t(B) * H * (T / 128);
    if (blocks <= size_t(std::min(T / 16 + 120, 200)))
        return BACKWARD_SPLIT;
    return blocks <= (T < 1024 ? 384 : 512) ? BACKWARD_BOTH : BACKWARD_IN_TURN;
}
void check_attention_shape(int B, int H, int T, int hd) {
    require(B > 0 && H > 0 && T > 0, "attention: empty shape");
    require(hd == HD, "attention: head_dim must be 64");
    require(T % 128 == 0, "attention: context must be a multiple of 128");
    require(size_t(B) * T < (size_t(1) << 31), "attention: too many tokens");
}
void check_matrix(const void *p, int ld, const char *name) {
    if (!p || (reinterpret_cast<uintptr_t>(p) & 15) || ld % 8)
        throw std::invalid_argument(std::string("attention operand ") + name +
                                    " must be non-null, 16-byte aligned, leading dimension % 8 == 0");
}

} // namespace

extern "C" int tgk_attn_fwd(hipStream_t stream, int B, int H, int T, int hd, const uint16_t *Q,
                            const uint16_t *K, const uint16_t *V, int ld, uint16_t *O, int ldo,
                            float *lse, float scale) {
    return guarded([&] {
        check_attention_shape(B, H, T, hd);
        check_matrix(Q, ld, "Q");
        check_matrix(K, ld, "K");
        check_matrix(V, ld, "V");
        check_matrix(O, ldo, "O");
        require(lse && !(reinterpret_cast<uintptr_t>(lse) & 15), "attention: lse must be 16-byte aligned");
        const bool split = forward_splits(B, H, T);
        const CausalGrid grid = split ? causal_grid(B, H, T, 32) : causal_grid(B, H, T, 128, 64);
        const auto kernel = !split ? attn_fwd_kernel : T > 128 ? attn_fwd_split_kernel<true> : attn_fwd_split_kernel<false>;
        hipLaunchKernelGGL(kernel, dim3(grid.blocks()), dim3(256), 0, stream, Q, K, V, ld, O, ldo, lse, T, grid, scale * LOG2E);
        check_hip(hipGetLastError(), "attention forward launch: ");
    });
}

extern "C" size_t tgk_attn_bwd_workspace(int B, int H, int T) {
    return 2 * size_t(B) * H * T * sizeof(float); // delta, and the log-sum-exp in base 2
}

namespace {
void attn_bwd_check(int B, int H, int T, int hd, const uint16_t *Q, const uint16_t *K, const uint16_t *V, int ld,
                    const uint16_t *O, int ldo, const float *lse, const uint16_t *dO, int lddo, uint16_t *dQ,
                    uint16_t *dK, uint16_t *dV, int lddq) {
    check_attention_shape(B, H, T, hd);
    check_matrix(Q, ld, "Q");
    check_matrix(K, ld, "K");
    check_matrix(V, ld, "V");
    check_matrix(O, ldo, "O");
    check_matrix(dO, lddo, "dO");
    check_matrix(dQ, lddq, "dQ");
    check_matrix(dK, lddq, "dK");
    check_matrix(dV, lddq, "dV");
    require(lse && !(reinterpret_cast<uintptr_t>(lse) & 15), "attention: lse must be 16-byte aligned");
}
// both backward kernels; `rows` holds delta[B*H*T] followed by the base-2 log-sum-exps[B*H*T]
void attn_bwd_launch(hipStream_t stream, int B, int H, int T, const uint16_t *Q, const uint16_t *K,
                     const uint16_t *V, int ld, const uint16_t *O, int ldo, const float *lse, const uint16_t *dO,
                     int lddo, uint16_t *dQ, uint16_t *dK, uint16_t *dV, int lddq, float scale, float *rows) {
    const Backward way = backward_way(B, H, T);
    if (way == BACKWARD_SPLIT) {
        const CausalGrid grid = causal_grid(B, H, T, 32);
        hipLaunchKernelGGL(attn_bwd_split_kernel, dim3(2 * grid.blocks()), dim3(256), 0, stream, Q, K, V, ld, dO, lddo, O, ldo,
                           lse, dQ, dK, dV, lddq, T, grid, scale);
        check_hip(hipGetLastError(), "attention backward launch: ");
        return;
    }
    float *delta = rows, *lse2 = delta + size_t(B) * H * T;
    const CausalGrid grid = causal_grid(B, H, T, 128);
    if (way == BACKWARD_BOTH) {
        hipLaunchKernelGGL(attn_delta_kernel, dim3(B * H * (T / 32)), dim3(256), 0, stream, dO, lddo, O, ldo, lse, lse2, delta, H, T);
        hipLaunchKernelGGL(attn_bwd_both_kernel, dim3(2 * grid.blocks()), dim3(256), 0, stream, Q, K, V, ld, dO, lddo, O, ldo,
                           lse, lse2, delta, dQ, dK, dV, lddq, T, grid, scale);
        check_hip(hipGetLastError(), "attention backward launch: ");
        return;
    }
    hipLaunchKernelGGL(attn_bwd_dq_kernel, dim3(grid.blocks()), dim3(256), 0, stream, Q, K, V, ld, dO, lddo, O, ldo, lse, lse2,
                       delta, dQ, lddq, T, grid, scale);
    hipLaunchKernelGGL(attn_bwd_dkdv_kernel, dim3(grid.blocks()), dim3(256), 0, stream, Q, K, V, ld, dO, lddo, lse2, delta, dK,
                       dV, lddq, T, grid, scale);
    check_hip(hipGetLastError(), "attention backward launch: ");
}
} // namespace

extern "C" int tgk_attn_bwd(hipStream_t stream, int B, int H, int T, int hd, const uint16_t *Q,
                            const uint16_t *K, const uint16_t *V, int ld, const uint16_t *O, int ldo,
                            const float *lse, const uint16_t *dO, int lddo, uint16_t *dQ, uint16_t *dK,
                            uint16_t *dV, int lddq, float scale, void *workspace,
                            size_t workspace_bytes) {
    return guarded([&] {
        attn_bwd_check(B, H, T, hd, Q, K, V, ld, O, ldo, lse, dO, lddo, dQ, dK, dV, lddq);
        require(workspace && workspace_bytes >= tgk_attn_bwd_workspace(B, H, T) &&
                    !(reinterpret_cast<uintptr_t>(workspace) & 15),
                "attention backward: workspace too small (see tgk_attn_bwd_workspace)");
        attn_bwd_launch(stream, B, H, T, Q, K, V, ld, O, ldo, lse, dO, lddo, dQ, dK, dV, lddq, scale,
                        static_cast<float *>(workspace));
    });
}

// ---- the same backward for callers that cannot allocate -------------------------------------------
// The two row vectors the kernels exchange (delta and the base-2 log-sum-exp, B*H*T floats each) live in
// a device array of this library instead of a caller's workspace.  Every GPU the library runs on holds
// its own copy of the array at its own address; the address is looked up once per device, with that
// device current, and only that address - never the array's name - is handed to kernels.  Every
// call writes the rows that it reads (dQ or attn_delta_kernel before dK/dV), so nothing has to be cleared between calls.
namespace {
constexpr size_t STATIC_BWD_ROWS = size_t(1) << 20; // B*H*T of one call: 8 MiB of device memory per GPU
static __device__ __align__(256) float scratch[2 * STATIC_BWD_ROWS];
constexpr int STATIC_MAX_DEVICES = 64;
std::atomic<float *> scratch_address[STATIC_MAX_DEVICES];

float *scratch_on_current_device() {
    int device = 0;
    check_hip(hipGetDevice(&device), "attention backward (static): ");
    require(device >= 0 && device < STATIC_MAX_DEVICES, "attention backward (static): device index out of range");
    float *address = scratch_address[device].load(std::memory_order_acquire);
    if (!address) {
        void *found = nullptr;
        check_hip(hipGetSymbolAddress(&found, HIP_SYMBOL(scratch)), "attention backward (static) scratch address: ");
        require(found != nullptr, "attention backward (static): the scratch array has no device address");
        address = static_cast<float *>(found);
        scratch_address[device].store(address, std::memory_order_release);
    }
    return address;
}
} // namespace

// Also the set-up call: it looks up the array's address on the current device, so that a later tgk_attn_bwd_static
// on this device (under stream capture, say) has nothing left to resolve.  A failed lookup is reported by that call.
extern "C" size_t tgk_attn_bwd_static_max_rows(void) {
    try {
        (void)scratch_on_current_device();
    } catch (const std::exception &) {
    }
    return STATIC_BWD_ROWS;
}

extern "C" int tgk_attn_bwd_static(hipStream_t stream, int B, int H, int T, int hd, const uint16_t *Q,
                                   const uint16_t *K, const uint16_t *V, int ld, const uint16_t *O, int ldo,
                                   const float *lse, const uint16_t *dO, int lddo, uint16_t *dQ, uint16_t *dK,
                                   uint16_t *dV, int lddq, float scale) {
    return guarded([&] {
        attn_bwd_check(B, H, T, hd, Q, K, V, ld, O, ldo, lse, dO, lddo, dQ, dK, dV, lddq);
        require(size_t(B) * H * T <= STATIC_BWD_ROWS,
                "attention backward (static): B*H*T exceeds tgk_attn_bwd_static_max_rows() = 1048576; "
                "use tgk_attn_bwd with a workspace");
        attn_bwd_launch(stream, B, H, T, Q, K, V, ld, O, ldo, lse, dO, lddo, dQ, dK, dV, lddq, scale,
                        scratch_on_current_device());
    });
}
