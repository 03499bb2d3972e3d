// The reference's own network behind the plain Config (config.h:4): width 16, 4 heads of 4, vocabulary
// 256, RMSNorm, partial RoPE, causal arg-max attention with a GELU gate, SwiGLU(48); optimizer pair
// mantissa-preserving AdamW + Muon.  Follows cuda/model.cuh:8-99 (op order and bf16 rounding points),
// cuda/ops.cuh:57-144, cuda/attention.cuh:4-106, cuda/optim.cuh:17-119.
//
// What bounds it is latency: a step is 1 GFLOP over some ten thousand tokens, and a sequence (at most eight positions)
// never leaves a wave.  So a wave takes sixteen tokens - whole sequences - through all layers in registers, forward and
// backward, with the weights in LDS as they are in memory.  Every factor of a product is a bf16 value, so products run on the
// bf16 matrix instructions, sixteen or thirty-two features at a time: 16 x 16 x 16 outputs are one instruction where the fp32 form
// takes four that wait for one another, and operands need no conversion.  Their sums are closer to 64 bits than a chain of fmaf in
// the features' order (normal factors, 16 / 48 / 256 terms: relative error 1.9e-8 / 3.7e-8 / 8.6e-8 against 2.2e-8 / 4.4e-8 /
// 1.07e-7), and an output depends on its own row and column alone, so results do not depend on how the tokens are cut.
// Lane 16 g + c holds features 4 g .. 4 g + 3 of token c: what such an instruction gives is what the next one takes, and head
// g of the token, one head a lane, so attention reads other positions' keys and values with DPP row shifts.
// Weight gradients are products over tokens: the waves of a block leave a layer's rows in LDS, the transposing load reads them
// across, and each wave sums some of the layer's tiles over the block's tokens; another launch adds the blocks' sums in order.
// No atomics, bit-reproducible (the place of weight_gradient's read-modify-write and of reduce_gradients,
// cuda/ops.cuh:83-109, cuda/trainer.cuh:9-47).
#include "common.h"
#include "width16.h"
#include "../../include/tgk_kernels.h"
#include <algorithm>
#include <atomic>
#include <type_traits>

// No product and sum is fused that is not written as fmaf: the kernels that share a function below have the same bits.
#pragma clang fp contract(off)

namespace {

constexpr int W = 16, HEADS = 4, F = 48, V = 256, MAX_DEPTH = 8;
constexpr int MAX_WAVES = 8; // waves of a block: they share the staged weights

struct Layer {
    int attention_norm, qkv, attention, mlp_norm, gate, up, down;
};
struct Layout { // model.h:12-37
    int embedding, final_norm, head, count;
    Layer layers[MAX_DEPTH];
};
constexpr int LAYER_SIZE = W + 3 * W * W + W * W + W + 3 * F * W;
__host__ __device__ inline Layer layer_layout(int l) {
    Layer b;
    b.attention_norm = V * W + l * LAYER_SIZE;
    b.qkv = b.attention_norm + W;
    b.attention = b.qkv + 3 * W * W;
    b.mlp_norm = b.attention + W * W;
    b.gate = b.mlp_norm + W;
    b.up = b.gate + F * W;
    b.down = b.up + F * W;
    return b;
}
Layout make_layout(int depth) {
    Layout p{};
    for (int l = 0; l < depth; ++l)
        p.layers[l] = layer_layout(l);
    p.embedding = 0;
    p.final_norm = V * W + depth * LAYER_SIZE;
    p.head = p.final_norm + W;
    p.count = p.head + V * W;
    return p;
}

// What a layer's forward pass keeps for its backward pass, 16 bytes a lane and slot: block input | post-attention residual,
// post-RoPE query | winning key, winning value | the two inverse norms, GELU(top) | GELU'(top) | distance to the winner, gate | up
// thrice, the gates' sigmoids thrice (cuda/types.cuh:40-44, cuda/model.cuh:25-29).  What else the backward pass wants it
// computes again: normalised rows, attention output and activation are a product of two of these each.
enum Slot { S_RESIDUAL, S_QUERY_KEY, S_VALUE_NORMS, S_GATE, S_GATE_UP, S_SIGMOID = S_GATE_UP + 3, SLOTS = S_SIGMOID + 3 };
struct Workspace {
    u32x4 *rows;               // [depth][waves][SLOTS][64]
    u32x2 *hidden, *nf;        // [waves][64], of the head
    float *inverse;            // [waves][64], of the final norm
    u32x2 *dlogits;            // [waves][16][64]
    float *partials;           // [blocks][parameters]
    int waves, blocks, waves_per_block;
    size_t bytes;
};
// another batch's, whose memory lies `apart` bytes further on
TG_DEVICE Workspace moved(Workspace s, int64_t apart) {
    const auto move = [&](auto *&p) { p = reinterpret_cast<std::remove_reference_t<decltype(p)>>(reinterpret_cast<char *>(p) + apart); };
    move(s.rows), move(s.hidden), move(s.nf), move(s.inverse), move(s.dlogits), move(s.partials);
    return s;
}
int tokens_per_wave(int context) { return 16 / context * context; }
// Four waves, one to a SIMD; eight where that fills more than the 256 units, whose LDS has room for one block each at depth 8: a
// step of 2304 sequences of 8 there 98 us with four, 75 with eight; of 10000 270 and 224; 4608 of 4 at depth 4 52 and 49.
int waves_per_block(int batch, int context) { return batch * context > tokens_per_wave(context) * 4 * 256 ? 8 : 4; }
int blocks_of(int batch, int context) {
    const int per_block = tokens_per_wave(context) * waves_per_block(batch, context);
    return (batch * context + per_block - 1) / per_block;
}
Workspace carve(int depth, int batch, int context, void *base) {
    Workspace r{};
    size_t at = 0;
    auto take = [&](size_t bytes) {
        void *p = base ? static_cast<unsigned char *>(base) + at : nullptr;
        at += (bytes + 255) & ~size_t(255);
        return p;
    };
    r.waves_per_block = waves_per_block(batch, context);
    r.blocks = blocks_of(batch, context);
    r.waves = r.blocks * r.waves_per_block;
    const size_t n = size_t(r.waves) * 64;
    r.rows = static_cast<u32x4 *>(take(n * depth * SLOTS * sizeof(u32x4)));
    r.hidden = static_cast<u32x2 *>(take(n * sizeof(u32x2)));
    r.nf = static_cast<u32x2 *>(take(n * sizeof(u32x2)));
    r.inverse = static_cast<float *>(take(n * sizeof(float)));
    r.dlogits = static_cast<u32x2 *>(take(n * 16 * sizeof(u32x2)));
    r.partials = static_cast<float *>(take(size_t(r.blocks) * make_layout(depth).count * sizeof(float)));
    r.bytes = at;
    return r;
}

// ---- device helpers ---------------------------------------------------------------------------------
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef short s16x8 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;

TG_DEVICE float master(const bf16_t *hi, const uint16_t *lo, int i) { // cuda/ops.cuh:6-9
    return __uint_as_float((uint32_t(hi[i]) << 16) | lo[i]);
}
TG_DEVICE u32x2 pack4(const f32x4 &v) {
    return u32x2{pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3])};
}
TG_DEVICE f32x4 unpack4(const u32x2 &t) {
    return f32x4{bf16_lo(t.x), bf16_hi(t.x), bf16_lo(t.y), bf16_hi(t.y)};
}
TG_DEVICE f32x4 rounded(const f32x4 &v) {
    return unpack4(pack4(v));
}
constexpr f32x4 ZERO = {0.f, 0.f, 0.f, 0.f};
TG_DEVICE float swap_add_16(float x) {
    const auto rows = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float(rows[0]) + __uint_as_float(rows[1]);
}
TG_DEVICE float swap_add_32(float x) {
    const auto halves = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float(halves[0]) + __uint_as_float(halves[1]);
}
TG_DEVICE float token_sum(const f32x4 &x) { // over a token's sixteen features
    return swap_add_32(swap_add_16((x[0] + x[1]) + (x[2] + x[3])));
}
TG_DEVICE float token_max(float x) { // over the four lanes that hold one token
    const auto rows = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    x = fmaxf(__uint_as_float(rows[0]), __uint_as_float(rows[1]));
    const auto halves = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return fmaxf(__uint_as_float(halves[0]), __uint_as_float(halves[1]));
}
// D[row][col] = sum over k of A[row][k] B[k][col] on top of acc, factors in bf16: lane 16 g + c gives A[c][4 g + j] and
// B[4 g + j][c] in element j and gets D[4 g + r][c] in register r; with two pairs of factors, k = 0 .. 15 of both.  A sum of three is
// two of the second form, with zeros: the first form right behind the second, adding to its result, gave wrong sums, and the
// compiler puts nothing between them.
TG_DEVICE f32x4 product(u32x2 a, u32x2 b, f32x4 acc = ZERO) {
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(s16x4, a), __builtin_bit_cast(s16x4, b), acc, 0, 0, 0);
}
TG_DEVICE f32x4 product(u32x2 a0, u32x2 b0, u32x2 a1, u32x2 b1, f32x4 acc = ZERO) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, u32x4{a0.x, a0.y, a1.x, a1.y}),
                                                   __builtin_bit_cast(bf16x8, u32x4{b0.x, b0.y, b1.x, b1.y}), acc, 0, 0, 0);
}
TG_DEVICE f32x4 product(u32x2 a0, u32x2 b0, u32x2 a1, u32x2 b1, u32x2 a2, u32x2 b2) {
    return product(a2, b2, u32x2{0, 0}, u32x2{0, 0}, product(a0, b0, a1, b1));
}
// the value of the lane D before / after this one in its row of sixteen (0 beyond the row)
template <int D> TG_DEVICE uint32_t earlier(uint32_t x) {
    if constexpr (D == 0)
        return x;
    else
        return uint32_t(__builtin_amdgcn_update_dpp(0, int(x), 0x110 + D, 0xF, 0xF, true));
}
template <int D> TG_DEVICE uint32_t later(uint32_t x) {
    if constexpr (D == 0)
        return x;
    else
        return uint32_t(__builtin_amdgcn_update_dpp(0, int(x), 0x100 + D, 0xF, 0xF, true));
}
template <int D, class Body> TG_DEVICE void from(Body &&body) { // D, D - 1, ..., 0
    body(std::integral_constant<int, D>{});
    if constexpr (D > 0)
        from<D - 1>(body);
}
template <int D, int END, class Body> TG_DEVICE void up_to(Body &&body) { // D, D + 1, ..., END
    body(std::integral_constant<int, D>{});
    if constexpr (D < END)
        up_to<D + 1, END>(body);
}
// 1 / b and x / b = divide(x, b, 1 / b), correctly rounded while neither b nor the result leaves the normal range (compared
// with the division over every mantissa of b and 262 million pairs: no difference): a Newton step on the hardware's
// approximate reciprocal, and for the quotient a correction by its residual, both with fused multiply-adds (Markstein, IBM
// Journal of Research and Development 34, 1990).  Three instructions where the division takes ten, and 140 of them stand in
// a wave's way at the head alone.
TG_DEVICE float reciprocal(float b) {
    const float r = __builtin_amdgcn_rcpf(b);
    return fmaf(fmaf(-b, r, 1.f), r, r);
}
TG_DEVICE float divide(float x, float b, float r) {
    const float q = x * r;
    return fmaf(fmaf(-q, b, x), r, q);
}
// e^x with the error of the library's (against 64 bits over (-87, 0) and (0, 88): 2.6e-8 of the value, at most 8.3e-8): 2^n times
// 2^f of the hardware, f within half of 0 and with what the rounding of x / ln 2 lost.  The bounds put in place of the library's
// two selections let infinities and NaN through the second term: ten instructions where it takes thirteen.
TG_DEVICE float exponential(float x) {
    constexpr float PER_LN2 = 1.44269504088896341f, REST = 1.92596299e-8f; // 1 / ln 2 in two parts
    const float t = __builtin_amdgcn_fmed3f(x * PER_LN2, -200.f, 200.f), n = rintf(t);
    return __builtin_amdgcn_ldexpf(__builtin_amdgcn_exp2f((t - n) + fmaf(x, REST, fmaf(x, PER_LN2, -t))), int(n));
}
// 1 / (1 + e^-x) taken 2^24 times too large, where the reciprocal stays in the normal range down to e^-x = 2^128; beyond that
// 2^-126 stands for it, which the last product rounds to 0.
TG_DEVICE float sigmoid(float x) {
    return reciprocal(fminf(fmaf(exponential(-x), 0x1p-24f, 0x1p-24f), 0x1p126f)) * 0x1p-24f;
}

struct Model {
    const bf16_t *hi;
    const uint16_t *lo;
    int depth, tokens, context, per_wave;
};
// a lane's place: token `token` (if `live`) at `position` of its sequence
struct Lane {
    int lane, c, g, wave, token, position;
    bool live;
};
template <int WAVES> TG_DEVICE Lane lane_of(const Model &m) {
    Lane p;
    p.lane = threadIdx.x & 63;
    p.c = p.lane & 15;
    p.g = p.lane >> 4;
    p.wave = blockIdx.x * WAVES + (threadIdx.x >> 6);
    p.token = p.wave * m.per_wave + p.c;
    p.live = p.c < m.per_wave && p.token < m.tokens;
    p.position = p.c % m.context;
    return p;
}

// A block's LDS: the weights' upper halves as they are in memory, from the embedding to the head, so that staging them is a
// copy and a token's row no further trip to memory behind the token's own; every RMSNorm scale in fp32; and for weight gradients
// each wave's rows, TILES tiles of 64 x 8 bytes in the lanes' order, its sums of the scales' gradients, and its tokens.
// Of a matrix of rows of 32 bytes a lane reads 8, operand of dX W^T; the transposing load gives it the operand of dY W.
constexpr int LAYER_BYTES = LAYER_SIZE * 2, QKV_AT = W * 2, ATTENTION_AT = QKV_AT + 3 * W * W * 2, GATE_AT = ATTENTION_AT + W * W * 2 + W * 2,
              UP_AT = GATE_AT + F * W * 2, DOWN_AT = UP_AT + F * W * 2, TILE = W * W * 2;
// of a layer; the head's dlogits and normalised rows, and the embedding's gradient, take their places
enum Tile { T_N1, T_A, T_N2, T_ACT, T_DQKV = T_ACT + 3, T_DH_ATTENTION = T_DQKV + 3, T_DGU, T_DH_DOWN = T_DGU + 6, TILES };
constexpr int T_DLOGITS = 0, T_NF = 16, T_DH = 0;
static_assert(TILES == 17, "the head's tiles fit a layer's");
__host__ __device__ constexpr int layer_at(int l) { return V * W * 2 + l * LAYER_BYTES; }
__host__ __device__ constexpr int head_at(int depth) { return layer_at(depth) + W * 2; }
__host__ __device__ constexpr int scales_at(int depth) { return head_at(depth) + V * W * 2; }
__host__ __device__ constexpr int rows_at(int depth) { return scales_at(depth) + (2 * depth + 1) * W * 4; }
__host__ __device__ constexpr int sums_at(int depth, int waves) { return rows_at(depth) + waves * TILES * 512; }
__host__ __device__ constexpr int ids_at(int depth, int waves) { return sums_at(depth, waves) + (2 * depth + 1) * waves * W * 4; }
__host__ __device__ constexpr int lds_bytes(int depth, int waves, bool gradients) {
    return gradients ? ids_at(depth, waves) + waves * 16 : rows_at(depth);
}
static_assert(layer_at(1) % 16 == 0 && head_at(1) % 16 == 0 && lds_bytes(MAX_DEPTH, MAX_WAVES, true) <= 160 * 1024, "LDS of a unit");

// `aligned` is false where the weights do not lie on 16 bytes
template <int WAVES> TG_DEVICE void stage(const Model &m, unsigned char *memory, bool aligned = true) {
    constexpr int THREADS = 64 * WAVES;
    const int bytes = scales_at(m.depth), wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (aligned) {
        const uint32_t lds = lds_address(memory) + uint32_t(wave * 1024);
        for (int at = 0; at < bytes; at += THREADS * 16) {
            const int mine = at + int(threadIdx.x) * 16;
            if (mine < bytes)
                async_copy16(lds + uint32_t(at), m.hi, uint32_t(mine));
        }
    } else {
#pragma unroll 4
        for (int at = int(threadIdx.x) * 8; at < bytes; at += THREADS * 8)
            *reinterpret_cast<u32x2 *>(memory + at) = *reinterpret_cast<const u32x2 *>(reinterpret_cast<const char *>(m.hi) + at);
    }
    float *scales = reinterpret_cast<float *>(memory + scales_at(m.depth));
    for (int at = threadIdx.x; at < (2 * m.depth + 1) * W; at += THREADS) {
        const int n = at >> 4; // attention and MLP norm of each layer, final
        const Layer q = layer_layout(n >> 1);
        const int offset = n == 2 * m.depth ? V * W + m.depth * LAYER_SIZE : (n & 1) ? q.mlp_norm : q.attention_norm;
        scales[at] = master(m.hi, m.lo, offset + (at & 15));
    }
    wait_vmcnt<0>();
    __syncthreads();
}
TG_DEVICE u32x2 read_across(const unsigned char *at) {
    return __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4 *)at));
}
// Lane 16 q + 4 j + m addresses eight bytes for a transposing load, and lane 16 q + i gets element i % 4 of what lanes
// 16 q + 4 * 0..3 + i / 4 address: with row 4 q + j, columns 4 m .. there, rows 4 q .. 4 q + 3 of column i.
struct Staged {
    const unsigned char *memory, *mine, *mine_down, *across, *across_down; // `down` has rows of 96 bytes
    const float *scales;
    int head;
    TG_DEVICE Staged(const Model &m, const unsigned char *memory_, const Lane &p) : memory(memory_) {
        const int row = 4 * p.g + ((p.lane >> 2) & 3), column = p.lane & 3;
        mine = memory + p.c * 32 + p.g * 8, mine_down = memory + DOWN_AT + p.c * 96 + p.g * 8;
        across = memory + row * 32 + column * 8, across_down = memory + DOWN_AT + row * 96 + column * 8;
        scales = reinterpret_cast<const float *>(memory + scales_at(m.depth)) + 4 * p.g;
        head = head_at(m.depth);
    }
    // operands of X W^T and of dY W: sixteen rows of a matrix; sixteen columns of `down`
    TG_DEVICE u32x2 operator()(int at) const { return *reinterpret_cast<const u32x2 *>(mine + at); }
    TG_DEVICE u32x2 down(int layer, int t) const { return *reinterpret_cast<const u32x2 *>(mine_down + layer + t * 32); }
    TG_DEVICE u32x2 turned(int at) const { return read_across(across + at); }
    TG_DEVICE u32x2 turned_down(int layer, int t) const { return read_across(across_down + layer + t * 32); }
    TG_DEVICE f32x4 scale(int norm) const { return *reinterpret_cast<const f32x4 *>(scales + norm * W); }
};

// cuda/ops.cuh:57-67: y = RN_bf16(v * rsqrt(mean(v^2) + 1e-6) * scale), scale read in full fp32
TG_DEVICE float inverse_rms(const f32x4 &v) {
    return __builtin_amdgcn_rsqf(token_sum(v * v) * (1.f / 16.f) + 1e-6f); // never denormal
}
// cuda/ops.cuh:68-80: the rounded input gradient of a row of inverse norm `inv` with z = v * inv
TG_DEVICE f32x4 normalize_backward(const f32x4 &z, float inv, const f32x4 &g, const f32x4 &scale) {
    const f32x4 dz = g * scale;
    const float dot = token_sum(dz * z);
    return rounded((dz - z * dot * (1.f / 16.f)) * inv);
}
// cuda/attention.cuh:19-30: first pair of every query and key head, one radian per position
TG_DEVICE void rotation(int position, float &c, float &s) {
    // float32(cos k), float32(sin k), k = 0..7 (cuda/attention.cuh:7-14)
    const float cos_table[8] = {1.0f, 0.5403022766113281f, -0.416146844625473f, -0.9899924993515015f,
                                -0.6536436080932617f, 0.28366219997406006f, 0.9601702690124512f, 0.7539022564888f};
    const float sin_table[8] = {0.0f, 0.8414709568023682f, 0.9092974066734314f, 0.14112000167369843f,
                                -0.756802499294281f, -0.9589242935180664f, -0.279415488243103f, 0.6569865942001343f};
    c = cos_table[0], s = sin_table[0];
#pragma unroll
    for (int k = 1; k < 8; ++k)
        if (position == k)
            c = cos_table[k], s = sin_table[k];
}
TG_DEVICE f32x4 rotate(f32x4 v, float c, float s) {
    const float x = v[0], y = v[1];
    v[0] = fmaf(x, c, -(y * s));
    v[1] = fmaf(x, s, y * c);
    return v;
}
TG_DEVICE f32x4 rotate_back(f32x4 v, float c, float s) {
    const float x = v[0], y = v[1];
    v[0] = fmaf(x, c, y * s);
    v[1] = fmaf(y, c, -(x * s));
    return v;
}

// Batches that share a launch: grid row y is member y's.  The members' workspaces are alike.
struct Group {
    W16Batch member[W16_BATCHES];
    TG_DEVICE Workspace workspace(const Workspace &first, int y) const {
        return moved(first, static_cast<const char *>(member[y].workspace) - static_cast<const char *>(member[0].workspace));
    }
};

// ---- forward ---------------------------------------------------------------------------------------
// What the head leaves for the backward pass; the logits' gradients in tiles of sixteen, but for the target's: lane g = target / 4
// % 4 has that (`at` in its own four of tile `tile`), the others none.
struct Head {
    u32x2 dlogits[16], hidden, nf;
    float inverse;
    bool holder;
    int tile, at;
    bf16_t of_target;
    // into a tile's four elements of this lane, behind the others
    template <class Place> TG_DEVICE void put(Place &&place) const {
#pragma unroll
        for (int t = 0; t < 16; ++t)
            *reinterpret_cast<u32x2 *>(place(t)) = dlogits[t];
        if (holder)
            reinterpret_cast<bf16_t *>(place(tile))[at] = of_target;
    }
};
TG_DEVICE f32x4 embedding_row(const unsigned char *memory, const Lane &p, int token) {
    return p.live ? unpack4(*reinterpret_cast<const u32x2 *>(memory + token * W * 2 + p.g * 8)) : ZERO;
}
// cuda/model.cuh:8-59.  dlogits = RN_bf16((p - onehot) / tokens).  GRADIENT: rows are kept in `s` and the head's in `head`.
template <bool GRADIENT, int CONTEXT>
TG_DEVICE void forward_pass(const Model &m, const Lane &p, const Staged &weight, const Workspace &s, f32x4 h, int target, float rc,
                            float rs, float *__restrict__ token_losses, float *__restrict__ logits_out, Head &head) {
    const int context = CONTEXT ? CONTEXT : m.context;
    for (int l = 0; l < m.depth; ++l) {
        const int at = layer_at(l);
        u32x4 *keep = s.rows + (size_t(l) * s.waves + p.wave) * SLOTS * 64 + p.lane;
        // QKV projection, RoPE (cuda/model.cuh:14-19)
        const float inv1 = inverse_rms(h);
        const u32x2 n1 = pack4(h * inv1 * weight.scale(2 * l));
        const f32x4 query = rounded(rotate(rounded(product(weight(at + QKV_AT), n1)), rc, rs));
        const u32x2 key = pack4(rotate(rounded(product(weight(at + QKV_AT + TILE), n1)), rc, rs));
        const u32x2 value = pack4(product(weight(at + QKV_AT + 2 * TILE), n1));
        // arg-max attention with its GELU gate (cuda/attention.cuh:33-71); keys in order, the first one wins ties
        float top = -INFINITY;
        int distance = 0;
        u32x2 best_key = {0, 0}, best_value = {0, 0};
        from<CONTEXT ? CONTEXT - 1 : 7>([&](auto step) {
            constexpr int D = decltype(step)::value;
            if (D >= context)
                return;
            const u32x2 k = {earlier<D>(key.x), earlier<D>(key.y)}, v = {earlier<D>(value.x), earlier<D>(value.y)};
            const f32x4 kf = unpack4(k);
            float score = 0.f;
#pragma unroll
            for (int c = 0; c < 4; ++c)
                score = fmaf(query[c], kf[c], score);
            const bool wins = D <= p.position && score > top;
            top = wins ? score : top;
            distance = wins ? D : distance;
            best_key.x = wins ? k.x : best_key.x, best_key.y = wins ? k.y : best_key.y;
            best_value.x = wins ? v.x : best_value.x, best_value.y = wins ? v.y : best_value.y;
        });
        const float e = 1.f + erff(top * 0.7071067811865475f);
        const float gate = 0.5f * top * e;
        const u32x2 a = pack4(unpack4(best_value) * gate);
        // output projection and residual: a bf16 add (cuda/model.cuh:20-21, cuda/mma.cuh:95-97)
        const f32x4 middle = rounded(rounded(product(weight(at + ATTENTION_AT), a)) + h);
        const float inv2 = inverse_rms(middle);
        const u32x2 n2 = pack4(middle * inv2 * weight.scale(2 * l + 1));
        if constexpr (GRADIENT) {
            const u32x2 x = pack4(h), mid = pack4(middle), q = pack4(query);
            keep[S_RESIDUAL * 64] = u32x4{x.x, x.y, mid.x, mid.y};
            keep[S_QUERY_KEY * 64] = u32x4{q.x, q.y, best_key.x, best_key.y};
            keep[S_VALUE_NORMS * 64] = u32x4{best_value.x, best_value.y, __float_as_uint(inv1), __float_as_uint(inv2)};
            const float slope = fmaf(top * 0.3989422804014327f, exponential(-0.5f * top * top), 0.5f * e);
            keep[S_GATE * 64] = u32x4{__float_as_uint(gate), __float_as_uint(slope), uint32_t(distance), 0};
        }
        // packed gate|up projection, SwiGLU (RN after SiLU and after the product), down projection and residual
        // (cuda/model.cuh:22-30, cuda/ops.cuh:120-131)
        u32x2 act[3];
#pragma unroll
        for (int t = 0; t < 3; ++t) {
            const u32x2 gate_row = pack4(product(weight(at + GATE_AT + t * TILE), n2)), up_row = pack4(product(weight(at + UP_AT + t * TILE), n2));
            const f32x4 x = unpack4(gate_row);
            f32x4 sig;
#pragma unroll
            for (int r = 0; r < 4; ++r)
                sig[r] = sigmoid(x[r]);
            act[t] = pack4(rounded(x * sig) * unpack4(up_row));
            if constexpr (GRADIENT) {
                keep[(S_GATE_UP + t) * 64] = u32x4{gate_row.x, gate_row.y, up_row.x, up_row.y};
                keep[(S_SIGMOID + t) * 64] = __builtin_bit_cast(u32x4, sig);
            }
        }
        const f32x4 out = product(weight.down(at, 0), act[0], weight.down(at, 1), act[1], weight.down(at, 2), act[2]);
        h = rounded(rounded(out) + middle);
    }
    // final RMSNorm, head, softmax cross-entropy (cuda/model.cuh:32-58): register r of tile t is logit 16 t + 4 g + r
    const float inv = inverse_rms(h);
    const u32x2 nf = pack4(h * inv * weight.scale(2 * m.depth));
    f32x4 logit[16];
    float high = -INFINITY;
#pragma unroll
    for (int t = 0; t < 16; ++t) {
        logit[t] = rounded(product(weight(weight.head + t * TILE), nf));
        high = fmaxf(fmaxf(high, fmaxf(logit[t][0], logit[t][1])), fmaxf(logit[t][2], logit[t][3]));
    }
    high = token_max(high);
    if (logits_out && p.live)
#pragma unroll
        for (int t = 0; t < 16; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                logits_out[size_t(p.token) * V + t * 16 + 4 * p.g + r] = logit[t][r];
    // the target's logit: tile target / 16, register target % 4 of the lane g = target / 4 % 4, by halves
    float of_four[16];
#pragma unroll
    for (int t = 0; t < 16; ++t) {
        const float even = target & 2 ? logit[t][2] : logit[t][0], odd = target & 2 ? logit[t][3] : logit[t][1];
        of_four[t] = target & 1 ? odd : even;
    }
#pragma unroll
    for (int bit = 0; bit < 4; ++bit)
#pragma unroll
        for (int t = 0; t < 8 >> bit; ++t)
            of_four[t] = target & (16 << bit) ? of_four[2 * t + 1] : of_four[2 * t];
    const bool holder = p.g == ((target >> 2) & 3);
    float picked = holder ? of_four[0] : 0.f;
#pragma unroll
    for (int t = 0; t < 16; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r)
            logit[t][r] = exponential(logit[t][r] - high);
    // the sum's tree: every 64th logit in order, then halves of what is left
    f32x4 quarter[4];
#pragma unroll
    for (int q = 0; q < 4; ++q)
        quarter[q] = ((logit[q] + logit[q + 4]) + logit[q + 8]) + logit[q + 12];
    const float sum = token_sum((quarter[0] + quarter[2]) + (quarter[1] + quarter[3]));
    picked = swap_add_16(swap_add_32(picked));
    if (p.live && p.g == 0)
        token_losses[p.token] = high + logf(sum) - picked;
    if constexpr (GRADIENT) {
        head.hidden = pack4(h), head.nf = nf, head.inverse = inv;
        // the quotient by sum * tokens in two parts: one rounding where two divisions have two
        const float tokens = float(m.tokens), whole = sum * tokens, share = reciprocal(whole);
        const float rest = share * fmaf(-fmaf(sum, tokens, -whole), share, fmaf(-whole, share, 1.f));
#pragma unroll
        for (int t = 0; t < 16; ++t) {
            f32x4 d;
#pragma unroll
            for (int r = 0; r < 4; ++r)
                d[r] = fmaf(logit[t][r], share, logit[t][r] * rest);
            const u32x2 packed = pack4(d);
            head.dlogits[t].x = p.live ? packed.x : 0, head.dlogits[t].y = p.live ? packed.y : 0;
        }
        const float probability = divide(exponential(picked - high), sum, reciprocal(sum));
        head.of_target = float_to_bf16(divide(probability - 1.f, tokens, 1.f / tokens));
        head.holder = holder && p.live, head.tile = target >> 4, head.at = target & 3;
    }
}

// ---- weight gradients ------------------------------------------------------------------------------
// A block sums what its waves kept in LDS over their tokens, in token order, tile by tile: partial[block].  The transposing load
// gives lane 16 q + i feature i of tokens 4 q .. 4 q + 3 of a wave, an operand of the instruction whose steps run over the
// tokens, two waves' tokens each.  That moves data and computes nothing: an infinity stays in its own feature.
template <int WAVES> struct Gradients {
    unsigned char *mine;         // this lane's place in this wave's tiles
    const unsigned char *across; // and in the first wave's, for the transposing load
    float *sums, *out;           // the waves' sums of the scales' gradients; partial[block]
    int c, g, wave;
    TG_DEVICE Gradients(const Model &m, unsigned char *memory, const Workspace &s, const Lane &p, int parameters)
        : c(p.c), g(p.g), wave(__builtin_amdgcn_readfirstlane(threadIdx.x >> 6)) {
        mine = memory + rows_at(m.depth) + wave * TILES * 512 + p.lane * 8;
        across = memory + rows_at(m.depth) + (16 * (p.lane & 3) + 4 * p.g + ((p.lane >> 2) & 3)) * 8;
        sums = reinterpret_cast<float *>(memory + sums_at(m.depth, WAVES));
        out = s.partials + size_t(blockIdx.x) * parameters;
    }
    TG_DEVICE void put(int tile, u32x2 row) const { *reinterpret_cast<u32x2 *>(mine + tile * 512) = row; }
    // sixteen rows of dW = dY^T X of `width` columns, sixteen of them
    TG_DEVICE void tile(int x, int dy, int at, int width) const {
        const auto row = [&](int n, int w) { return read_across(across + (w * TILES + n) * 512); };
        f32x4 sum = ZERO;
#pragma unroll
        for (int w = 0; w < WAVES; w += 2)
            sum = product(row(x, w), row(dy, w), row(x, w + 1), row(dy, w + 1), sum);
        *reinterpret_cast<f32x4 *>(out + at + c * width + 4 * g) = sum;
    }
    TG_DEVICE void layer(int l) const {
        const Layer q = layer_layout(l);
        // thirteen tiles
        constexpr int HALVES = WAVES / 4;
        const int part = wave / HALVES, half = HALVES == 1 ? -1 : wave % HALVES; // a half: the first two tiles or the rest
        const auto mine_too = [&](int n) { return half < 0 || half == (n >= 2); };
        if (part == 0) {
#pragma unroll
            for (int t = 0; t < 3; ++t)
                if (mine_too(t))
                    tile(T_N1, T_DQKV + t, q.qkv + t * W * W, W);
            if (mine_too(3))
                tile(T_A, T_DH_ATTENTION, q.attention, W);
        } else if (part == 3) {
#pragma unroll
            for (int t = 0; t < 3; ++t)
                if (mine_too(t))
                    tile(T_ACT + t, T_DH_DOWN, q.down + t * W, F);
        } else {
#pragma unroll
            for (int t = 0; t < 3; ++t)
                if (mine_too(t))
                    tile(T_N2, T_DGU + 3 * (part - 1) + t, (part == 1 ? q.gate : q.up) + t * W * W, W);
        }
    }
    TG_DEVICE void head(int depth) const {
#pragma unroll
        for (int t = 0; t < 16 / WAVES; ++t)
            tile(T_NF, T_DLOGITS + wave * (16 / WAVES) + t, V * W + depth * LAYER_SIZE + W + (wave * (16 / WAVES) + t) * W * W, W);
    }
    // the terms g * z of a norm's scale, over this wave's tokens
    TG_DEVICE void scale(int norm, f32x4 terms) const {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const auto turn = [&](auto by) {
                terms[r] += __uint_as_float(uint32_t(__builtin_amdgcn_update_dpp(0, int(__float_as_uint(terms[r])), 0x120 + decltype(by)::value, 0xF, 0xF, true)));
            };
            turn(std::integral_constant<int, 8>{}), turn(std::integral_constant<int, 4>{}), turn(std::integral_constant<int, 2>{}), turn(std::integral_constant<int, 1>{});
        }
        if (c == 0)
            *reinterpret_cast<f32x4 *>(sums + (norm * WAVES + wave) * W + 4 * g) = terms;
    }
    TG_DEVICE void scales(int depth) const {
        for (int at = threadIdx.x; at < (2 * depth + 1) * W; at += 64 * WAVES) {
            const int norm = at >> 4;
            float sum = 0.f;
#pragma unroll
            for (int w = 0; w < WAVES; ++w)
                sum += sums[(norm * WAVES + w) * W + (at & 15)];
            const Layer q = layer_layout(norm >> 1);
            out[(norm == 2 * depth ? V * W + depth * LAYER_SIZE : (norm & 1) ? q.mlp_norm : q.attention_norm) + (at & 15)] = sum;
        }
    }
    // The embedding's rows: the one-hot matrix of the tokens times the gradient.  0 times an infinity is NaN, in ids that have
    // no part in it, so where a row is not finite the rows are added one by one.
    TG_DEVICE void embedding(const unsigned char *ids) const {
        constexpr int N = V / 16 / WAVES; // tiles of sixteen ids
        const int first = wave * N * 16 + c;
        f32x4 sum[N];
        bool extreme = false;
#pragma unroll
        for (int n = 0; n < N; ++n)
            sum[n] = ZERO;
#pragma unroll
        for (int w = 0; w < WAVES; w += 2) {
            u32x2 rows[2];
            uint32_t four[2];
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                rows[k] = read_across(across + ((w + k) * TILES + T_DH) * 512);
                four[k] = *reinterpret_cast<const uint32_t *>(ids + (w + k) * 16 + 4 * g);
                const auto either = [](uint32_t two) { return (two & 0x7f80u) == 0x7f80u || (two & 0x7f800000u) == 0x7f800000u; };
                extreme = extreme || either(rows[k].x) || either(rows[k].y);
            }
#pragma unroll
            for (int n = 0; n < N; ++n) {
                u32x2 hot[2];
#pragma unroll
                for (int k = 0; k < 2; ++k) {
                    const auto one = [&](int j) { return int((four[k] >> (8 * j)) & 255u) == first + n * 16; };
                    hot[k].x = (one(0) ? 0x3f80u : 0u) | (one(1) ? 0x3f800000u : 0u);
                    hot[k].y = (one(2) ? 0x3f80u : 0u) | (one(3) ? 0x3f800000u : 0u);
                }
                sum[n] = product(rows[0], hot[0], rows[1], hot[1], sum[n]);
            }
        }
        if (__builtin_amdgcn_ballot_w64(extreme)) {
#pragma unroll
            for (int n = 0; n < N; ++n)
                sum[n] = ZERO;
#pragma unroll 1
            for (int t = 0; t < WAVES * 16; ++t) {
                const int w = t >> 4, id = ids[t];
                const f32x4 row = unpack4(*reinterpret_cast<const u32x2 *>(mine + ((w - wave) * TILES + T_DH) * 512 + ((t & 15) - c) * 8));
#pragma unroll
                for (int n = 0; n < N; ++n)
                    if (id == first + n * 16)
                        sum[n] = sum[n] + row;
            }
        }
#pragma unroll
        for (int n = 0; n < N; ++n)
            *reinterpret_cast<f32x4 *>(out + (first + n * 16) * W + 4 * g) = sum[n];
    }
};

// ---- backward --------------------------------------------------------------------------------------
// cuda/model.cuh:61-99
template <int CONTEXT, int WAVES>
TG_DEVICE void backward_pass(const Model &m, const Lane &p, const Staged &weight, const Workspace &s, float rc, float rs,
                             const Head &head, unsigned char *memory, int token, int parameters) {
    const int context = CONTEXT ? CONTEXT : m.context;
    const Gradients<WAVES> gradients(m, memory, s, p, parameters);
    unsigned char *ids = memory + ids_at(m.depth, WAVES);

    // a layer's rows are requested while the layer above is worked on
    struct Rows {
        u32x4 slot[SLOTS];
    };
    auto request = [&](int l, Rows &r) {
        const u32x4 *keep = s.rows + (size_t(l) * s.waves + p.wave) * SLOTS * 64 + p.lane;
#pragma unroll
        for (int i = 0; i < SLOTS; ++i)
            r.slot[i] = keep[i * 64];
    };

    // head input gradient and final RMSNorm backward (cuda/model.cuh:63-66)
    Rows next;
    request(m.depth - 1, next);
    if (p.g == 0)
        ids[gradients.wave * 16 + p.c] = uint8_t(token);
    f32x4 dn = ZERO;
    head.put([&](int t) { return gradients.mine + (T_DLOGITS + t) * 512; });
    gradients.put(T_NF, head.nf);
    const auto dlogits = [&](int t) { return *reinterpret_cast<const u32x2 *>(gradients.mine + (T_DLOGITS + t) * 512); };
#pragma unroll
    for (int t = 0; t < 16; t += 2)
        dn = product(weight.turned(weight.head + t * TILE), dlogits(t), weight.turned(weight.head + (t + 1) * TILE), dlogits(t + 1), dn);
    const f32x4 z = unpack4(head.hidden) * head.inverse;
    dn = rounded(dn);
    gradients.scale(2 * m.depth, dn * z);
    f32x4 dh = normalize_backward(z, head.inverse, dn, weight.scale(2 * m.depth));
    __syncthreads();
    gradients.head(m.depth);
    for (int l = m.depth - 1; l >= 0; --l) {
        const int at = layer_at(l);
        const Rows rows = next;
        if (l)
            request(l - 1, next);
        // down projection, SwiGLU, packed gate|up projection and RMSNorm backward (cuda/model.cuh:72-88, cuda/ops.cuh:133-144)
        u32x2 packed = pack4(dh), act[3], dgate[3], dup[3];
#pragma unroll
        for (int t = 0; t < 3; ++t) {
            const u32x4 gu = rows.slot[S_GATE_UP + t];
            const f32x4 gate = unpack4(u32x2{gu.x, gu.y}), up = unpack4(u32x2{gu.z, gu.w}), sig = __builtin_bit_cast(f32x4, rows.slot[S_SIGMOID + t]);
            const f32x4 dy = rounded(product(weight.turned_down(at, t), packed)), da = rounded(dy * up), silu = rounded(gate * sig);
            f32x4 d;
#pragma unroll
            for (int r = 0; r < 4; ++r)
                d[r] = da[r] * sig[r] * fmaf(gate[r], 1.f - sig[r], 1.f);
            dgate[t] = pack4(d), dup[t] = pack4(dy * silu), act[t] = pack4(silu * up);
        }
        __syncthreads(); // the tiles above this layer's have been read
        gradients.put(T_DH_DOWN, packed);
#pragma unroll
        for (int t = 0; t < 3; ++t)
            gradients.put(T_ACT + t, act[t]), gradients.put(T_DGU + t, dgate[t]), gradients.put(T_DGU + 3 + t, dup[t]);
        const auto gate_at = [&](int t) { return weight.turned(at + GATE_AT + t * TILE); }; // up's tiles lie behind
        dn = product(gate_at(4), dup[1], gate_at(5), dup[2],
                     product(gate_at(2), dgate[2], gate_at(3), dup[0], product(gate_at(0), dgate[0], gate_at(1), dgate[1])));
        dn = rounded(dn);
        const u32x4 residual = rows.slot[S_RESIDUAL], value_norms = rows.slot[S_VALUE_NORMS];
        const float inv1 = __uint_as_float(value_norms.z), inv2 = __uint_as_float(value_norms.w);
        const f32x4 z2 = unpack4(u32x2{residual.z, residual.w}) * inv2, scale2 = weight.scale(2 * l + 1);
        gradients.put(T_N2, pack4(z2 * scale2));
        gradients.scale(2 * l + 1, dn * z2);
        // residual gradients stay bf16 between operators (cuda/ops.cuh:74-76)
        dh = rounded(dh + normalize_backward(z2, inv2, dn, scale2));
        packed = pack4(dh);
        gradients.put(T_DH_ATTENTION, packed);

        // attention: output projection backward, the score gradient of the cached winner, query / key / value gradients
        // gathered over the sequence, inverse RoPE, QKV projection and RMSNorm backward (cuda/model.cuh:89-96,
        // cuda/attention.cuh:72-106)
        const u32x4 query_key = rows.slot[S_QUERY_KEY];
        const u32x2 query = {query_key.x, query_key.y};
        const f32x4 key = unpack4(u32x2{query_key.z, query_key.w}), value = unpack4(u32x2{value_norms.x, value_norms.y});
        const float gate = __uint_as_float(rows.slot[S_GATE].x), slope = __uint_as_float(rows.slot[S_GATE].y);
        const uint32_t distance = rows.slot[S_GATE].z;
        gradients.put(T_A, pack4(value * gate));
        const u32x2 dattn = pack4(product(weight.turned(at + ATTENTION_AT), packed));
        const f32x4 da = unpack4(dattn);
        float dt = 0.f;
#pragma unroll
        for (int c = 0; c < 4; ++c)
            dt = fmaf(da[c], value[c], dt);
        dt *= slope;
        f32x4 dk = ZERO, dv = ZERO;
        up_to<0, CONTEXT ? CONTEXT - 1 : 7>([&](auto step) { // queries of this token's sequence that chose it, in order
            constexpr int D = decltype(step)::value;
            if (D >= context)
                return;
            // every lane takes part in the shifts, so none of them may sit behind a condition
            const uint32_t theirs = later<D>(distance);
            const float their_dt = __uint_as_float(later<D>(__float_as_uint(dt))), their_gate = __uint_as_float(later<D>(__float_as_uint(gate)));
            const f32x4 qf = unpack4(u32x2{later<D>(query.x), later<D>(query.y)});
            const f32x4 df = unpack4(u32x2{later<D>(dattn.x), later<D>(dattn.y)});
            // skipped, not multiplied by 0: what did not choose this token may be infinite
            if (p.position + D < context && theirs == uint32_t(D)) {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    dk[r] = fmaf(their_dt, qf[r], dk[r]);
                    dv[r] = fmaf(df[r], their_gate, dv[r]);
                }
            }
        });
        const u32x2 dq_row = pack4(rotate_back(rounded(key * dt), rc, rs)), dk_row = pack4(rotate_back(rounded(dk), rc, rs)), dv_row = pack4(dv);
        gradients.put(T_DQKV, dq_row), gradients.put(T_DQKV + 1, dk_row), gradients.put(T_DQKV + 2, dv_row);
        dn = product(weight.turned(at + QKV_AT), dq_row, weight.turned(at + QKV_AT + TILE), dk_row, weight.turned(at + QKV_AT + 2 * TILE), dv_row);
        dn = rounded(dn);
        const f32x4 z1 = unpack4(u32x2{residual.x, residual.y}) * inv1, scale1 = weight.scale(2 * l);
        gradients.put(T_N1, pack4(z1 * scale1));
        gradients.scale(2 * l, dn * z1);
        dh = rounded(dh + normalize_backward(z1, inv1, dn, scale1));
        __syncthreads();
        gradients.layer(l);
    }
    __syncthreads();
    gradients.put(T_DH, pack4(dh));
    __syncthreads();
    gradients.embedding(ids);
    gradients.scales(m.depth);
}

// ---- kernels -----------------------------------------------------------------------------------------
template <bool GRADIENT, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void w16_forward_kernel(Model m, const uint8_t *__restrict__ x, const uint8_t *__restrict__ y,
                                                               Workspace s, float *__restrict__ token_losses,
                                                               float *__restrict__ logits_out) {
    extern __shared__ __align__(16) unsigned char memory[];
    const Lane p = lane_of<WAVES>(m);
    const Staged weight(m, memory, p);
    const int token = p.live ? x[p.token] : 0, target = p.live ? y[p.token] : 0;
    stage<WAVES>(m, memory, !(reinterpret_cast<uintptr_t>(m.hi) & 15));
    const f32x4 h = embedding_row(memory, p, token);
    float rc, rs;
    rotation(p.position, rc, rs);
    Head head;
    forward_pass<GRADIENT, 0>(m, p, weight, s, h, target, rc, rs, token_losses, logits_out, head);
    if constexpr (GRADIENT) {
        const size_t here = size_t(p.wave) * 64 + p.lane;
        s.hidden[here] = head.hidden, s.nf[here] = head.nf, s.inverse[here] = head.inverse;
        head.put([&](int t) { return s.dlogits + (size_t(p.wave) * 16 + t) * 64 + p.lane; });
    }
}
template <int WAVES>
__global__ __launch_bounds__(64 * WAVES) void w16_backward_kernel(Model m, const uint8_t *__restrict__ x, Workspace s, int parameters) {
    extern __shared__ __align__(16) unsigned char memory[];
    const Lane p = lane_of<WAVES>(m);
    const Staged weight(m, memory, p);
    const int token = p.live ? x[p.token] : 0;
    Head head;
    const size_t here = size_t(p.wave) * 64 + p.lane;
    head.hidden = s.hidden[here], head.nf = s.nf[here], head.inverse = s.inverse[here];
#pragma unroll
    for (int t = 0; t < 16; ++t)
        head.dlogits[t] = s.dlogits[(size_t(p.wave) * 16 + t) * 64 + p.lane];
    head.holder = false; // the target's is among them
    stage<WAVES>(m, memory, !(reinterpret_cast<uintptr_t>(m.hi) & 15));
    float rc, rs;
    rotation(p.position, rc, rs);
    backward_pass<0, WAVES>(m, p, weight, s, rc, rs, head, memory, token, parameters);
}
// A training step's both passes: a wave's backward pass reads only what its own forward pass kept, so the two are one launch
// and the weights are staged once.  What bounds it is a wave's chain of some 1100 dependent vector instructions a layer and 1200 at
// the head.  Depth 4, 2560 sequences of 4: 38.7 us on fp32 matrix instructions, weights converted on the way, without the weight
// gradients, which took 13.1 us more from rows kept in memory; 24.6 so.  Depth 8, 16 of 8: 64.9 + 11.1 and 39.0.  Tokens and
// targets come straight out of the training bytes, every sequence a window at a hashed place (cuda/dataset.cuh:13-27).
template <int CONTEXT, int WAVES>
__global__ __launch_bounds__(64 * WAVES) __attribute__((amdgpu_waves_per_eu(2, 2))) void w16_step_kernel(
    Model m, W16Data data, uint64_t inverse, Workspace first, Group group, int parameters) {
    extern __shared__ __align__(16) unsigned char memory[];
    const W16Batch &batch = group.member[blockIdx.y];
    const Workspace s = group.workspace(first, blockIdx.y);
    m.hi = batch.weights.hi, m.lo = batch.weights.lo;
    const Lane p = lane_of<WAVES>(m);
    const Staged weight(m, memory, p);
    int token = 0, target = 0;
    if (p.live) {
        const int sequence = p.token / CONTEXT;
        // the hash modulo the places: `inverse` is 2^64 / places rounded down, so the quotient is at most one too small
        const uint64_t hash = hash_u64(data.seed + batch.step * uint64_t(m.tokens / CONTEXT) + uint64_t(sequence));
        const uint64_t low = 8, places = uint64_t(data.size) - low;
        uint64_t place = hash - __umul64hi(hash, inverse) * places;
        place -= place >= places ? places : 0;
        const int64_t end = int64_t(low + place);
        const uint8_t *window = data.bytes + (end - CONTEXT) + p.position;
        token = window[0], target = window[1];
    }
    stage<WAVES>(m, memory);
    const f32x4 h = embedding_row(memory, p, token);
    float rc, rs;
    rotation(p.position, rc, rs);
    Head head;
    forward_pass<true, CONTEXT>(m, p, weight, s, h, target, rc, rs, batch.token_losses, nullptr, head);
    backward_pass<CONTEXT, WAVES>(m, p, weight, s, rc, rs, head, memory, token, parameters);
}

// ---- the blocks' sums --------------------------------------------------------------------------------
// gradient = the blocks' sums in block order, in up to GROUPS parts: a wave takes 64 elements, GROUPS waves share out the blocks,
// and a part's loads are in flight together.  160 blocks of 21648 parameters: 8.2 us with one wave for 64 elements, 5.2 so; of 2
// blocks (35088 parameters, four batches) eight waves make 7.5 and one 4.8: up to sixteen blocks take one.
// Where norms are wanted, every wave's elements leave a part of a sum of squares of 1024 (FOLD_PARTS).
// Blocks beyond the parameters average the losses: one a position, in double (cuda/trainer.cuh:79-100).
constexpr int FOLD_PARTS = 1024 / 64;
int fold_parts(int parameters) { return (parameters + 1023) / 1024 * FOLD_PARTS; }
template <int GROUPS>
__global__ __launch_bounds__(GROUPS == 1 ? 256 : 64 * GROUPS) void w16_fold_kernel(Workspace whole, Group group, int parameters, int blocks,
                                                                                 int batch, int context) {
    constexpr int WAVES = GROUPS == 1 ? 4 : GROUPS;
    const W16Batch &member = group.member[blockIdx.y];
    const int count = whole.blocks, lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (int(blockIdx.x) >= blocks) {
        __shared__ double sums[WAVES];
        const int position = blockIdx.x - blocks;
        double sum = 0;
#pragma unroll 4
        for (int b = threadIdx.x; b < batch; b += 64 * WAVES)
            sum += member.token_losses[size_t(b) * context + position];
#pragma unroll
        for (int k = 32; k; k >>= 1)
            sum += __shfl_xor(sum, k, 64);
        if (lane == 0)
            sums[wave] = sum;
        __syncthreads();
        if (threadIdx.x == 0) {
            sum = sums[0];
            for (int w = 1; w < WAVES; ++w)
                sum += sums[w];
            member.means[position] = float(sum / batch);
        }
        return;
    }
    const int part = GROUPS == 1 ? blockIdx.x * WAVES + wave : blockIdx.x, at = part * 64 + lane;
    const int share = (count + GROUPS - 1) / GROUPS, first = GROUPS == 1 ? 0 : wave * share, mine = min(share, count - first);
    float sum = 0.f;
    if (at < parameters) {
        const float *from = group.workspace(whole, blockIdx.y).partials + size_t(first) * parameters + at;
        constexpr int AT_ONCE = GROUPS == 1 ? 8 : 20;
        for (int c = 0; c < mine; c += AT_ONCE) {
            float v[AT_ONCE];
#pragma unroll
            for (int i = 0; i < AT_ONCE; ++i)
                if (c + i < mine)
                    v[i] = from[size_t(c + i) * parameters];
#pragma unroll
            for (int i = 0; i < AT_ONCE; ++i)
                if (c + i < mine)
                    sum += v[i];
        }
    }
    if constexpr (GROUPS > 1) {
        __shared__ float rows[GROUPS][64];
        rows[wave][lane] = sum;
        __syncthreads();
        if (wave)
            return;
        sum = rows[0][lane];
#pragma unroll
        for (int w = 1; w < GROUPS; ++w)
            sum += rows[w][lane];
    }
    if (at < parameters)
        member.gradient[at] = sum;
    if (!member.norms)
        return;
    const float squares = wave_sum(sum * sum);
    if (lane == 0)
        member.norms[part] = squares;
}

// ---- optimizer (cuda/optim.cuh:17-119) ------------------------------------------------------------------
// Blocks 0 .. 5 depth - 1: Muon, a hidden matrix each.  The rest: AdamW, 256 quads of embedding, scales and head each.
// The Newton-Schulz iterate is a 16 x n matrix of bf16 values in 16 x 16 tiles, one a wave, lane 16 g + c holding rows 4 g .. of
// column c.  X X^T is symmetric to the last bit, so what a lane holds of it is the operand of the two products behind it, every
// wave computes it for itself, and a step exchanges nothing but X through LDS: one barrier a step.  What bounds it is that chain:
// 8.6 us a launch on fp32 matrix instructions, 5.5 more for every further step; on the bf16 ones, with the clip factors of all
// steps formed at the start, 6.8 and 3.0.
// One launch makes as many steps, one after another, as there are gradients at hand: an element's (Muon: a matrix's) weights
// and state stay in the registers between them.
struct Update {
    float *momentum, *variance;
    int norm_count, norm_parts, depth; // norms: norm_count sums of norm_parts partial sums each, 1 or FOLD_PARTS
    int count;
    W16Step step[W16_BATCHES];
};
// The steps' clip factors, a step a wave: clip_factor of the norms.  A barrier stands between this and their first use.
TG_DEVICE void clip_factors(const Update &u, float *factors) {
    const int lane = threadIdx.x & 63;
    for (int n = threadIdx.x >> 6; n < u.count; n += 4) {
        const W16Step &step = u.step[n];
        float factor = 1.f;
        if (step.adam.clip > 0.f) {
            float sum = 0.f;
            if (u.norm_parts == 1)
                for (int i = lane; i < u.norm_count; i += 64)
                    sum += step.norms[i];
            else
                for (int i = lane; i < u.norm_count * FOLD_PARTS / 4; i += 64) {
                    const f32x4 part = reinterpret_cast<const f32x4 *>(step.norms)[i];
                    sum += (part[0] + part[1]) + (part[2] + part[3]);
                }
            factor = fminf(1.f, step.adam.clip / (sqrtf(wave_sum(sum)) + 1e-6f));
        }
        if (lane == 0)
            factors[n] = factor;
    }
}
TG_DEVICE void muon_matrix(const Update &u, int matrix, float *factors) {
    __shared__ __align__(8) bf16_t wide[2][16 * F];
    __shared__ float norm_waves[2][4];
    const Layer p = layer_layout(matrix / 5);
    const int type = matrix % 5;
    const int weight = type == 0 ? p.qkv : type == 1 ? p.attention : type == 2 ? p.gate : type == 3 ? p.up : p.down;
    const int rows = (type == 0 || type == 2 || type == 3) ? 48 : 16, cols = type == 4 ? 48 : 16;
    const int n = rows > cols ? rows : cols, size = rows * cols, tid = threadIdx.x;
    // element tid + 256 k of the matrix is this thread's until the iteration and again behind it; its place in the 16 x n form
    auto place = [&](int i) { return rows > cols ? (i % cols) * rows + i / cols : i; };
    float next_g[3], m[3], w[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const int i = weight + tid + 256 * k;
        const bool mine = tid + 256 * k < size;
        next_g[k] = mine ? u.step[0].gradient[i] : 0.f, m[k] = mine ? u.momentum[i] : 0.f;
        w[k] = mine ? master(u.step[0].from.hi, u.step[0].from.lo, i) : 0.f;
    }
    clip_factors(u, factors);
    __syncthreads();
    const int lane = tid & 63, c = lane & 15, gr = lane >> 4, tile = tid >> 6, tiles = n / 16;
    for (int at = 0; at < u.count; ++at) {
        const W16Step &u_step = u.step[at];
        const MuonArgs &muon = u_step.muon;
        const float g[3] = {next_g[0], next_g[1], next_g[2]};
        if (at + 1 < u.count)
#pragma unroll
            for (int k = 0; k < 3; ++k)
                next_g[k] = tid + 256 * k < size ? u.step[at + 1].gradient[weight + tid + 256 * k] : 0.f;
        const float clip = factors[at];
        float squares = 0.f, b[3];
#pragma unroll
        for (int k = 0; k < 3; ++k)
            if (tid + 256 * k < size) {
                const float gs = g[k] * clip;
                m[k] = fmaf(1.f - muon.momentum, fmaf(g[k], clip, -m[k]), m[k]);
                b[k] = round_bf16(fmaf(muon.momentum, m[k] - gs, gs));
                squares = fmaf(b[k], b[k], squares);
            }
        const float norm = fmaxf(round_bf16(sqrtf(block_sum_256(squares, norm_waves[at & 1]))), round_bf16(1e-7f));
#pragma unroll
        for (int k = 0; k < 3; ++k)
            if (tid + 256 * k < size)
                wide[0][place(tid + 256 * k)] = float_to_bf16(b[k] / norm);
        __syncthreads();
        f32x4 x = ZERO; // rows 4 gr .. of column 16 tile + c
        if (tile < tiles)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                x[r] = bf16_to_float(wide[0][(4 * gr + r) * n + 16 * tile + c]);
        for (int step = 0; step < muon.ns_steps; ++step) {
            const bf16_t *in = wide[step & 1] + c * n + 4 * gr;
            bf16_t *out = wide[(step & 1) ^ 1] + 4 * gr * n + 16 * tile + c;
            if (tile < tiles) {
                const auto row = [&](int k) { return *reinterpret_cast<const u32x2 *>(in + 16 * k); };
                const u32x2 first = row(0);
                f32x4 gram; // A = X X^T, kept in bf16
                if (tiles == 1)
                    gram = product(first, first);
                else {
                    const u32x2 second = row(1), third = row(2);
                    gram = product(first, first, second, second, third, third);
                }
                const u32x2 gram_row = pack4(gram);
                gram = unpack4(gram_row);
                const f32x4 square = product(gram_row, gram_row);
                f32x4 work; // -4.775 A + 2.0315 A A
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    work[r] = fmaf(2.0315f, square[r], -4.775f * gram[r]);
                const f32x4 change = product(pack4(work), pack4(x));
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    x[r] = fmaf(3.4445f, x[r], change[r]);
                const u32x2 packed = pack4(x);
                x = unpack4(packed);
                out[0] = bf16_t(packed.x), out[n] = bf16_t(packed.x >> 16);
                out[2 * n] = bf16_t(packed.y), out[3 * n] = bf16_t(packed.y >> 16);
            }
            __syncthreads();
        }
        const bf16_t *result = wide[muon.ns_steps & 1];
        const float adjusted = muon.lr * sqrtf(fmaxf(1.f, float(rows) / float(cols))), keep = fmaf(-muon.lr, muon.weight_decay, 1.f);
#pragma unroll
        for (int k = 0; k < 3; ++k)
            if (tid + 256 * k < size) {
                const int i = weight + tid + 256 * k;
                w[k] = fmaf(w[k], keep, -(adjusted * bf16_to_float(result[place(tid + 256 * k)])));
                const uint32_t bits = __float_as_uint(w[k]);
                u_step.to.hi[i] = uint16_t(bits >> 16); // cuda/ops.cuh:10-14
                u_step.to.lo[i] = uint16_t(bits);
            }
        __syncthreads(); // the next step's matrix goes where this one's result is read
    }
#pragma unroll
    for (int k = 0; k < 3; ++k)
        if (tid + 256 * k < size)
            u.momentum[weight + tid + 256 * k] = m[k];
}
__global__ __launch_bounds__(256) void w16_update_kernel(Update u) {
    __shared__ float factors[W16_BATCHES];
    if (int(blockIdx.x) < 5 * u.depth)
        return muon_matrix(u, blockIdx.x, factors);
    // quads: the embedding's 1024, four for each scale, the head's 1024 (the only ones that decay)
    const int quad = (blockIdx.x - 5 * u.depth) * 256 + threadIdx.x, norm = (quad - V * W / 4) >> 2, norms = 2 * u.depth + 1;
    int at = quad * 4;
    bool decays = false, live = true;
    if (norm >= norms) {
        const int k = quad - V * W / 4 - 4 * norms;
        live = k < V * W / 4;
        at = live ? V * W + u.depth * LAYER_SIZE + W + k * 4 : 0;
        decays = true;
    } else if (norm >= 0 && quad >= V * W / 4) {
        const Layer q = layer_layout(norm >> 1);
        at = (norm == 2 * u.depth ? V * W + u.depth * LAYER_SIZE : (norm & 1) ? q.mlp_norm : q.attention_norm) + (quad & 3) * 4;
    }
    f32x4 m = *reinterpret_cast<const f32x4 *>(u.momentum + at), v = *reinterpret_cast<const f32x4 *>(u.variance + at), w;
#pragma unroll
    for (int k = 0; k < 4; ++k)
        w[k] = master(u.step[0].from.hi, u.step[0].from.lo, at + k);
    f32x4 next_g = *reinterpret_cast<const f32x4 *>(u.step[0].gradient + at);
    clip_factors(u, factors);
    __syncthreads();
    if (!live)
        return;
    for (int n = 0; n < u.count; ++n) {
        const W16Step &step = u.step[n];
        const f32x4 g = next_g;
        if (n + 1 < u.count)
            next_g = *reinterpret_cast<const f32x4 *>(u.step[n + 1].gradient + at);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            float mk = m[k], vk = v[k];
            w[k] = adamw_element(step.adam, decays ? step.adam.weight_decay : 0.f, factors[n], w[k], mk, vk, g[k]);
            m[k] = mk, v[k] = vk;
        }
        const auto half = [&](int k, int shift) { return (__float_as_uint(w[k]) >> shift) & 0xffffu; };
        *reinterpret_cast<u32x2 *>(step.to.hi + at) = u32x2{half(0, 16) | half(1, 16) << 16, half(2, 16) | half(3, 16) << 16};
        *reinterpret_cast<u32x2 *>(step.to.lo + at) = u32x2{half(0, 0) | half(1, 0) << 16, half(2, 0) | half(3, 0) << 16};
    }
    *reinterpret_cast<f32x4 *>(u.momentum + at) = m;
    *reinterpret_cast<f32x4 *>(u.variance + at) = v;
}
int adam_blocks(int depth) { return (2 * V * W / 4 + 4 * (2 * depth + 1) + 255) / 256; }

void check_shape(int depth, int batch, int context) {
    require(depth >= 1 && depth <= MAX_DEPTH, "w16: depth must be 1..8");
    require(context >= 1 && context <= 8, "w16: context must be 1..8 (the RoPE table has eight entries)");
    require(batch >= 1, "w16: empty batch");
    require(int64_t(batch) * context <= (1 << 24), "w16: too many tokens");
}
Model make_model(int depth, int batch, int context, const uint16_t *hi, const uint16_t *lo) {
    return Model{hi, lo, depth, batch * context, context, tokens_per_wave(context)};
}

} // namespace

extern "C" int tgk_w16_parameter_count(int depth) {
    return depth >= 1 && depth <= MAX_DEPTH ? make_layout(depth).count : 0;
}

extern "C" size_t tgk_w16_workspace(int depth, int batch, int context) {
    if (depth < 1 || depth > MAX_DEPTH || batch < 1 || context < 1 || context > 8)
        return 0;
    return carve(depth, batch, context, nullptr).bytes;
}

namespace {
// the kernels' LDS beyond 64 KiB is a per-device attribute
template <class Kernel> void allow_lds(Kernel kernel, std::atomic<bool> (&configured)[64], size_t bytes) {
    int device = 0;
    check_hip(hipGetDevice(&device));
    require(device >= 0 && device < 64, "w16: device index out of range");
    if (configured[device].load(std::memory_order_acquire))
        return;
    check_hip(hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, int(bytes)),
              "w16 LDS size: ");
    configured[device].store(true, std::memory_order_release);
}
void launch_fold(hipStream_t stream, const Model &m, const Workspace &r, const Group &group, int count, bool losses) {
    const int parameters = make_layout(m.depth).count;
    const bool many = r.blocks > 16;
    const int blocks = many ? fold_parts(parameters) : fold_parts(parameters) / 4;
    hipLaunchKernelGGL(many ? w16_fold_kernel<8> : w16_fold_kernel<1>, dim3(blocks + (losses ? m.context : 0), count), dim3(many ? 512 : 256), 0,
                       stream, r, group, parameters, blocks, m.tokens / m.context, m.context);
    check_hip(hipGetLastError(), "w16 fold launch: ");
}
} // namespace

extern "C" int tgk_w16_forward(hipStream_t stream, int depth, int batch, int context, const uint16_t *weight_hi,
                               const uint16_t *weight_lo, const uint8_t *x, const uint8_t *y, void *workspace,
                               float *token_losses, float *logits, int with_gradient) {
    return guarded([&] {
        check_shape(depth, batch, context);
        require(weight_hi && weight_lo && x && y && workspace && token_losses, "w16_forward: missing operand");
        require(!(reinterpret_cast<uintptr_t>(workspace) & 255), "w16_forward: workspace must be 256-byte aligned");
        const Model m = make_model(depth, batch, context, weight_hi, weight_lo);
        const Workspace r = carve(depth, batch, context, workspace);
        static std::atomic<bool> configured[4][64];
        const bool wide = r.waves_per_block == 8;
        const auto kernel = with_gradient ? (wide ? w16_forward_kernel<true, 8> : w16_forward_kernel<true, 4>)
                                          : (wide ? w16_forward_kernel<false, 8> : w16_forward_kernel<false, 4>);
        allow_lds(kernel, configured[2 * (with_gradient != 0) + wide], lds_bytes(MAX_DEPTH, r.waves_per_block, false));
        hipLaunchKernelGGL(kernel, dim3(r.blocks), dim3(64 * r.waves_per_block), lds_bytes(depth, r.waves_per_block, false), stream, m, x, y, r,
                           token_losses, logits);
        check_hip(hipGetLastError(), "w16_forward launch: ");
    });
}

extern "C" int tgk_w16_backward(hipStream_t stream, int depth, int batch, int context, const uint16_t *weight_hi,
                                const uint16_t *weight_lo, const uint8_t *x, void *workspace, float *gradient) {
    return guarded([&] {
        check_shape(depth, batch, context);
        require(weight_hi && weight_lo && x && workspace && gradient, "w16_backward: missing operand");
        require(!(reinterpret_cast<uintptr_t>(workspace) & 255), "w16_backward: workspace must be 256-byte aligned");
        const Model m = make_model(depth, batch, context, weight_hi, weight_lo);
        const Workspace r = carve(depth, batch, context, workspace);
        static std::atomic<bool> configured[2][64];
        const bool wide = r.waves_per_block == 8;
        const auto kernel = wide ? w16_backward_kernel<8> : w16_backward_kernel<4>;
        allow_lds(kernel, configured[wide], lds_bytes(MAX_DEPTH, r.waves_per_block, true));
        hipLaunchKernelGGL(kernel, dim3(r.blocks), dim3(64 * r.waves_per_block), lds_bytes(depth, r.waves_per_block, true), stream, m, x, r,
                           make_layout(depth).count);
        check_hip(hipGetLastError(), "w16_backward launch: ");
        Group group{};
        group.member[0].workspace = workspace, group.member[0].gradient = gradient;
        launch_fold(stream, m, r, group, 1, false);
    });
}

int w16_blocks(int batch, int context) {
    return blocks_of(batch, context);
}
int w16_norm_count(int depth) {
    return fold_parts(make_layout(depth).count) / FOLD_PARTS;
}
int w16_norm_parts() {
    return FOLD_PARTS;
}
void w16_gradients(hipStream_t stream, int depth, int batch, int context, const W16Data &data, int count, const W16Batch *batches) {
    require(context == 4 || context == 8, "w16: a training step has a context of 4 or 8");
    require(count >= 1 && count <= W16_BATCHES, "w16: too many batches for one launch");
    const Model m = make_model(depth, batch, context, nullptr, nullptr);
    const Workspace r = carve(depth, batch, context, batches[0].workspace);
    Group group{};
    std::copy(batches, batches + count, group.member);
    static std::atomic<bool> configured[4][64];
    const bool wide = r.waves_per_block == 8;
    const auto kernel = context == 4 ? (wide ? w16_step_kernel<4, 8> : w16_step_kernel<4, 4>) : (wide ? w16_step_kernel<8, 8> : w16_step_kernel<8, 4>);
    allow_lds(kernel, configured[2 * (context == 8) + wide], lds_bytes(MAX_DEPTH, r.waves_per_block, true));
    const uint64_t places = uint64_t(data.size) - 8, inverse = places > 1 ? uint64_t((static_cast<unsigned __int128>(1) << 64) / places) : ~uint64_t(0);
    hipLaunchKernelGGL(kernel, dim3(r.blocks, count), dim3(64 * r.waves_per_block), lds_bytes(depth, r.waves_per_block, true), stream, m, data,
                       inverse, r, group, make_layout(depth).count);
    check_hip(hipGetLastError(), "w16_step launch: ");
    launch_fold(stream, m, r, group, count, true);
}
void w16_updates(hipStream_t stream, int depth, float *momentum, float *variance, int norm_count, int norm_parts, int count,
                 const W16Step *steps) {
    require(count >= 1 && count <= W16_BATCHES, "w16: too many steps for one launch");
    Update u{momentum, variance, norm_count, norm_parts, depth, count, {}};
    std::copy(steps, steps + count, u.step);
    hipLaunchKernelGGL(w16_update_kernel, dim3(5 * depth + adam_blocks(depth)), dim3(256), 0, stream, u);
    check_hip(hipGetLastError(), "w16_update launch: ");
}

extern "C" int tgk_w16_muon(hipStream_t stream, int depth, uint16_t *weight_hi, uint16_t *weight_lo, float *momentum,
                            const float *gradient, const float *norm_partials, int norm_count, float clip, float lr,
                            float momentum_rate, float weight_decay, int ns_steps) {
    return guarded([&] {
        require(depth >= 1 && depth <= MAX_DEPTH, "w16_muon: depth must be 1..8");
        require(weight_hi && weight_lo && momentum && gradient, "w16_muon: missing operand");
        require(!(clip > 0.f) || (norm_partials && norm_count > 0), "w16_muon: clipping needs the norm partials");
        require(ns_steps >= 1 && ns_steps <= 10, "w16_muon: ns_steps must be 1..10");
        AdamArgs adam{};
        adam.clip = clip;
        const W16Weights weights{weight_hi, weight_lo};
        Update u{momentum, nullptr, norm_count, 1, depth, 1, {}};
        u.step[0] = {weights, weights, gradient, norm_partials, adam, MuonArgs{lr, momentum_rate, weight_decay, ns_steps}};
        hipLaunchKernelGGL(w16_update_kernel, dim3(5 * depth), dim3(256), 0, stream, u); // the matrices' blocks alone
        check_hip(hipGetLastError(), "w16_muon launch: ");
    });
}
