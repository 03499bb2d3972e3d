// The reference's own network behind the plain Config (config.h:4): width 16, 4 heads of 4, vocabulary
// 256, RMSNorm, partial RoPE, causal arg-max attention with a GELU gate, SwiGLU(48); optimizer pair
// mantissa-preserving AdamW + Muon.  Follows cuda/model.cuh:8-99 (op order and bf16 rounding points),
// cuda/ops.cuh:57-144, cuda/attention.cuh:4-106, cuda/optim.cuh:17-119.
//
// What bounds it is latency: a step is 1 GFLOP over some ten thousand tokens, and a sequence (at most eight positions)
// never leaves a team.  So a team of four waves takes sixteen tokens - whole sequences - through all layers in registers and LDS,
// forward and backward, with the weights staged in LDS as matrix operands.  Products run on
// v_mfma_f32_16x16x4_f32, which is bit for bit a chain of fmaf over its four k (measured on random and extreme values;
// the bf16 forms add in an order of their own): every sum has one order, the k's own, whatever the kernel's shape, so
// results do not depend on how the work is cut.  This instruction takes 32 cycles in which its SIMD does no vector arithmetic,
// of no wave (measured); of that a lone wave issues one instruction in five cycles, two waves two.  Lane 16 g + c works for token c:
//   "feed" layout: register j holds feature 4 j + g - what step j of a product over features wants from that lane;
//   "head" layout: register r holds feature 4 g + r - head g of the token, one head a lane, so attention reads other
//   positions' keys and values with DPP row shifts.
// A product's results come out in either, by the order of the weight's rows.  Weight gradients are products over tokens,
// another launch: a block for the rows that one layer kept of a chunk of tokens, which the transposing load reads across,
// so that a chain of fmaf runs over the tokens in order; one more folds the chunks in order.  No atomics, bit-reproducible
// (the place of weight_gradient's read-modify-write and of reduce_gradients, cuda/ops.cuh:83-109, cuda/trainer.cuh:9-47).
#include "common.h"
#include "width16.h"
#include "width16_launch.h"
#include "../../include/tgk_kernels.h"
#include <algorithm>
#include <atomic>
#include <type_traits>

// No product and sum is fused that is not written as fmaf: the kernels that share a function below have the same bits.
#pragma clang fp contract(off)

namespace {

using namespace w16;
constexpr int HEADS = 4, F = 48;
constexpr int WAVES = 4;       // waves of a block of weight gradients, whose chunks are whole numbers of four teams' tokens
constexpr int CHUNK_WAVES = 8; // waves' tokens in one partial sum of a weight gradient (128 tokens)

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

// Rows that a team leaves for the weight gradients, tiles of 64 x 8 bytes in the lanes' own order, side by side: normalised
// rows, attention output, activation, and the gradients that are their other operands.
enum Tile { T_N1, T_A, T_N2, T_ACT, T_DQKV = T_ACT + 3, T_DH_ATTENTION = T_DQKV + 3, T_DGU, T_DH_DOWN = T_DGU + 6, OPERANDS };
constexpr int ROW_FEATURES = ROW_BYTES, LONE_ROW_BYTES = ROW_FEATURES + 6 * 512; // a lone wave keeps gate and up there, too
struct Workspace {
    u32x2 *tiles;        // [depth][waves][OPERANDS][64]
    unsigned char *rows; // [depth][waves][LONE_ROW_BYTES], where they do not stay in LDS
    float *gz;       // [2 depth + 1][waves * 16][16]: g * z of every RMSNorm scale; the final norm's last
    u32x2 *hidden, *nf, *dh; // [waves][64]
    float *inverse;  // [waves][64] of the final norm
    u32x2 *dlogits;  // [waves][16][64]
    float *partials; // [chunks][parameters]
    int waves, blocks, chunks;
    size_t bytes;
};
// another batch's, whose memory lies `apart` bytes further on
TG_DEVICE Workspace moved(Workspace s, int64_t apart) {
    const auto move = [&](auto *&p) { p = reinterpret_cast<std::remove_reference_t<decltype(p)>>(reinterpret_cast<char *>(p) + apart); };
    move(s.tiles), move(s.rows), move(s.gz), move(s.hidden), move(s.nf), move(s.dh), move(s.inverse), move(s.dlogits), move(s.partials);
    return s;
}
int tokens_per_wave(int context) { return 16 / context * context; }
int blocks_of(int batch, int context) {
    const int per_block = tokens_per_wave(context) * WAVES;
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
    r.blocks = blocks_of(batch, context);
    r.waves = r.blocks * WAVES;
    r.chunks = (r.waves + CHUNK_WAVES - 1) / CHUNK_WAVES;
    const size_t n = size_t(r.waves) * 64;
    r.tiles = static_cast<u32x2 *>(take(n * depth * OPERANDS * sizeof(u32x2)));
    r.rows = static_cast<unsigned char *>(take(size_t(r.waves) * depth * LONE_ROW_BYTES));
    r.gz = static_cast<float *>(take(n * (2 * depth + 1) * 4 * sizeof(float)));
    r.hidden = static_cast<u32x2 *>(take(n * sizeof(u32x2)));
    r.nf = static_cast<u32x2 *>(take(n * sizeof(u32x2)));
    r.dh = static_cast<u32x2 *>(take(n * sizeof(u32x2)));
    r.inverse = static_cast<float *>(take(n * sizeof(float)));
    r.dlogits = static_cast<u32x2 *>(take(n * 16 * sizeof(u32x2)));
    r.partials = static_cast<float *>(take(size_t(r.chunks) * make_layout(depth).count * sizeof(float)));
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
// These values are worked out here and not further on.
template <class T> TG_DEVICE void ready(T &value) {
    asm volatile("" : "+v"(value));
}
template <class T, class... More> TG_DEVICE void ready(T &value, More &...more) {
    ready(value);
    ready(more...);
}
// No vector arithmetic moves across; memory and scalar instructions may.
TG_DEVICE void products_only() {
    __builtin_amdgcn_sched_barrier(0x4 | 0x10 | 0x80);
}
// D[row][col] = fmaf chain over k = 0 .. 15 of A[row][k] B[k][col], on top of acc: lane 16 g + c gives A[c][4 j + g] and
// B[4 j + g][c] in register j and gets D[4 g + r][c] in register r.  The four instructions stand together: a wave's vector arithmetic
// and this form of product take turns, 33 cycles a product in a chain, but 50 with the next one's operand made between them.
TG_DEVICE f32x4 multiply(f32x4 a, f32x4 b, f32x4 acc = ZERO) {
    ready(a, b);
    products_only();
#pragma unroll
    for (int j = 0; j < 4; ++j)
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[j], b[j], acc, 0, 0, 0);
    products_only();
    return acc;
}
// N products with the same second operand
template <int N> TG_DEVICE void multiply_all(f32x4 (&a)[N], f32x4 b, f32x4 (&product)[N]) {
#pragma unroll
    for (int n = 0; n < N; ++n)
        ready(a[n]), product[n] = ZERO;
    ready(b);
    products_only();
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int n = 0; n < N; ++n)
            product[n] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[n][j], b[j], product[n], 0, 0, 0);
    products_only();
}
TG_DEVICE float swap_add_16(float x) {
    const auto rows = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float(rows[0]) + __uint_as_float(rows[1]);
}
TG_DEVICE float swap_add_32(float x) {
    const auto halves = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float(halves[0]) + __uint_as_float(halves[1]);
}
TG_DEVICE float token_max(float x) { // over the four lanes that hold one token
    const auto rows = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    x = fmaxf(__uint_as_float(rows[0]), __uint_as_float(rows[1]));
    const auto halves = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return fmaxf(__uint_as_float(halves[0]), __uint_as_float(halves[1]));
}
// head layout <-> feed layout: the 4 x 4 transposition of (lane group, register)
TG_DEVICE f32x4 turned(const f32x4 &v) {
    const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(v[0]), __float_as_uint(v[2]), false, false);
    const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v[1]), __float_as_uint(v[3]), false, false);
    const auto c = __builtin_amdgcn_permlane16_swap(a[0], b[0], false, false);
    const auto d = __builtin_amdgcn_permlane16_swap(a[1], b[1], false, false);
    return f32x4{__uint_as_float(c[0]), __uint_as_float(c[1]), __uint_as_float(d[0]), __uint_as_float(d[1])};
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
// e^-x for a bf16 value x, bit for bit expf's over all of them: log2(e) in sixteen bits times x is exact, so that what the
// rounding to a power of two leaves is, too, and one fused step brings the rest.  Beyond +-200 the result is 0 or infinite.
TG_DEVICE float exp_of_minus(float x) {
    const float y = __builtin_amdgcn_fmed3f(-x, -200.f, 200.f), t = y * 1.44268798828125f, n = __builtin_rintf(t);
    return __builtin_amdgcn_ldexpf(__builtin_amdgcn_exp2f(fmaf(y, 7.052607713e-06f, t - n)), int(n));
}
// 1 / (1 + e^-x) of a bf16 value, taken 2^24 times too large, where the reciprocal stays in the normal range down to
// e^-x = 2^128; beyond that 2^-126 stands for it, which the last product rounds to 0.  (Of NaN any value: it is multiplied by x.)
TG_DEVICE float sigmoid(float x) {
    return reciprocal(fminf(fmaf(exp_of_minus(x), 0x1p-24f, 0x1p-24f), 0x1p126f)) * 0x1p-24f;
}

struct Model {
    const bf16_t *hi;
    const uint16_t *lo;
    int depth, tokens, context, per_wave;
    int teams; // of a block
};
// a lane's place: token `token` (if `live`) at `position` of its sequence, in the team `wave` of the batch, of which its wave
// has the role `role`
struct Lane {
    int lane, c, g, wave, role, team, token, position;
    bool live;
};
// Consecutive waves of a block sit on consecutive SIMDs: the teams' first roles, which have the longest way, on different ones.
// A team beyond the batch's last repeats that one.
template <int R = ROLES> TG_DEVICE Lane lane_of(const Model &m, int waves) {
    Lane p;
    const int at = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    p.lane = threadIdx.x & 63;
    p.c = p.lane & 15;
    p.g = p.lane >> 4;
    p.team = at / R;
    p.role = (at + p.team) % R;
    p.wave = min(int(blockIdx.x) * m.teams + p.team, waves - 1);
    p.token = p.wave * m.per_wave + p.c;
    p.live = p.c < m.per_wave && p.token < m.tokens;
    p.position = p.c % m.context;
    return p;
}

TG_DEVICE int feed_row(int row) { return ((row & 3) << 2) | (row >> 2); } // its own inverse
// Byte offset, in a tile of items (g, c), of the item that lane 16 q + 4 j + m addresses for a transposing load: (m, 4 q + j)
// or (m, 4 j + q).  Lane 16 q + i then gets element i % 4 of items (i / 4, 4 q + 0..3) or (i / 4, 4 * 0..3 + q).
TG_DEVICE int across_offset(int lane, bool natural) {
    const int q = lane >> 4, j = (lane >> 2) & 3, m = lane & 3;
    return (16 * m + (natural ? 4 * j + q : 4 * q + j)) * 8;
}
TG_DEVICE u32x2 read_across(const unsigned char *at) {
    return __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4 *)at));
}
// Of n waves, wave w stages tiles w, w + n, ... of every layer and of the head: all loads go out before the first is waited for,
// and every address is a layer's away from the one before.
template <int R = ROLES> struct Staging {
    static constexpr int WAVES = block_waves(R), PER_LAYER = (LAYER_TILES + WAVES - 1) / WAVES, HEADS = HEAD_TILES / WAVES;
    static_assert(WAVES * 64 >= (2 * MAX_DEPTH + 1) * W && HEADS * WAVES == HEAD_TILES && V * W * 2 <= WAVES * 1024,
                  "every scale has a thread, every tile a wave, every KiB of the embedding one");
    const Model &m;
    unsigned char *tiles;
    u32x2 v[PER_LAYER][MAX_DEPTH], head[HEADS];
    float scale;
    int lane, wave;
    TG_DEVICE Staging(const Model &m_, unsigned char *memory)
        : m(m_), tiles(memory), lane(threadIdx.x & 63), wave(__builtin_amdgcn_readfirstlane(threadIdx.x >> 6)) {}
    TG_DEVICE float *scales() const { return reinterpret_cast<float *>(tiles + staged_tiles(m.depth) * 512); }
    // a lane brings four elements of one row: k = 4 (lane % 4) .. + 3
    TG_DEVICE int row_offset(int width) const { return (lane >> 2) * width + (lane & 3) * 4; }
    TG_DEVICE static int tile_offset(int k) { // of tile k in its layer's weights
        const Layer q = layer_layout(0);
        return k < 4 ? q.qkv + k * 256 : k < 10 ? q.gate + (k - 4) * 256 : q.down + (k - 10) * 16;
    }
    TG_DEVICE void request() {
#pragma unroll
        for (int i = 0; i < PER_LAYER; ++i) {
            const int k = wave + i * WAVES;
            if (k >= LAYER_TILES)
                break;
            const bf16_t *from = m.hi + tile_offset(k) + (k < 10 ? row_offset(W) : row_offset(F)); // rows of `down` are 48 long
#pragma unroll
            for (int l = 0; l < MAX_DEPTH; ++l) // a layer beyond the last is the last again
                v[i][l] = *reinterpret_cast<const u32x2 *>(from + min(l, m.depth - 1) * LAYER_SIZE);
        }
#pragma unroll
        for (int i = 0; i < HEADS; ++i)
            head[i] = *reinterpret_cast<const u32x2 *>(m.hi + V * W + m.depth * LAYER_SIZE + W + row_offset(W) + (wave + i * WAVES) * 256);
        const int n = threadIdx.x >> 4; // attention and MLP norm of each layer, final
        const Layer q = layer_layout(n >> 1);
        const int offset = n == 2 * m.depth ? V * W + m.depth * LAYER_SIZE : (n & 1) ? q.mlp_norm : q.attention_norm;
        if (n <= 2 * m.depth)
            scale = master(m.hi, m.lo, offset + (threadIdx.x & 15));
    }
    // 8 KiB, 16 bytes a lane of the last eight waves; `aligned` is false where the weights are not
    TG_DEVICE void request_embedding(bool aligned = true) const {
        unsigned char *to = tiles + embedding_at(m.depth);
        const int piece = wave - (WAVES - V * W * 2 / 1024);
        if (!aligned)
            for (int i = threadIdx.x; i < V * W / 4; i += WAVES * 64)
                reinterpret_cast<u32x2 *>(to)[i] = reinterpret_cast<const u32x2 *>(m.hi)[i];
        else if (piece >= 0)
            async_copy16(lds_address(to) + uint32_t(piece * 1024), m.hi, uint32_t(piece * 1024 + lane * 16));
    }
    TG_DEVICE static uint16_t element(const u32x2 &v, int e) { return uint16_t((e < 2 ? v.x : v.y) >> ((e & 1) * 16)); }
    // element e of a lane's four is k = 4 j + e: item (e, row), element j.  `to`: the lane's place in the tile
    TG_DEVICE static void put(unsigned char *to, const u32x2 &v) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
            *reinterpret_cast<uint16_t *>(to + e * 128) = element(v, e);
    }
    TG_DEVICE void finish(bool backward) {
        const int row = lane >> 2, j = lane & 3;
        unsigned char *natural = tiles + row * 8 + j * 2, *feed = tiles + feed_row(row) * 8 + j * 2;
        // the attention projection again: rows = inputs 4 j + e, k = output `row`: item (row % 4, input), element row / 4
        unsigned char *turned = tiles + (m.depth * LAYER_TILES + HEAD_TILES) * 512 + ((row & 3) * 16 + 4 * j) * 8 + (row >> 2) * 2;
#pragma unroll
        for (int i = 0; i < PER_LAYER; ++i) {
            const int k = wave + i * WAVES;
            if (k >= LAYER_TILES)
                break;
            unsigned char *to = (k > 2 ? feed : natural) + k * 512;
#pragma unroll
            for (int l = 0; l < MAX_DEPTH; ++l) {
                if (l >= m.depth)
                    break;
                put(to + l * LAYER_TILES * 512, v[i][l]);
                if (backward && k == 3)
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        *reinterpret_cast<uint16_t *>(turned + l * 512 + e * 8) = element(v[i][l], e);
            }
        }
#pragma unroll
        for (int i = 0; i < HEADS; ++i)
            put(feed + (m.depth * LAYER_TILES + wave + i * WAVES) * 512, head[i]);
        if (int(threadIdx.x) < (2 * m.depth + 1) * W)
            scales()[threadIdx.x] = scale;
        wait_vmcnt<0>(); // the embedding
        __syncthreads();
    }
    // whether this wave is in a team; the others have done their part
    TG_DEVICE bool stays() const { return wave < m.teams * R; }
};
struct Staged {
    const unsigned char *tiles;
    const float *scales;
    int lane, g, head, turned_attention; // tiles: the head's first, the first attention projection for the backward pass
    int feed, natural; // across_offset
    TG_DEVICE Staged(const Model &m, const unsigned char *memory, const Lane &p)
        : tiles(memory), scales(reinterpret_cast<const float *>(memory + staged_tiles(m.depth) * 512)), lane(p.lane), g(p.g),
          head(m.depth * LAYER_TILES), turned_attention(head + HEAD_TILES), feed(across_offset(p.lane, false)),
          natural(across_offset(p.lane, true)) {}
    TG_DEVICE f32x4 operator()(int tile) const { return unpack4(*reinterpret_cast<const u32x2 *>(tiles + tile * 512 + lane * 8)); }
    // the transposed operand, of a tile in feed order or (q, k, v) in the matrix's own
    TG_DEVICE u32x2 turned_feed_row(int tile) const { return read_across(tiles + tile * 512 + feed); }
    TG_DEVICE f32x4 turned_feed(int tile) const { return unpack4(turned_feed_row(tile)); }
    TG_DEVICE f32x4 turned_natural(int tile) const { return unpack4(read_across(tiles + tile * 512 + natural)); }
    TG_DEVICE f32x4 scale(int norm) const {
        const float *s = scales + norm * W + g;
        return f32x4{s[0], s[4], s[8], s[12]};
    }
};

// feed-layout rows times feed-layout rows of the same token, an fmaf chain in feature order: the diagonal of a product
TG_DEVICE float token_dot(const f32x4 &a, const f32x4 &b, const Lane &p) {
    const f32x4 all = multiply(a, b);
    float mine = 0.f;
#pragma unroll
    for (int r = 0; r < 4; ++r)
        mine = 4 * p.g + r == p.c ? all[r] : mine;
    return swap_add_32(swap_add_16(mine)); // the other three lanes hold zeros
}
// cuda/ops.cuh:57-67: y = RN_bf16(v * rsqrt(mean(v^2) + 1e-6) * scale), scale read in full fp32
TG_DEVICE float inverse_rms(const f32x4 &v, const Lane &p) {
    const float sum = token_dot(v, v, p);
    return rsqrtf(sum * (1.f / 16.f) + 1e-6f);
}
TG_DEVICE u32x2 normalize(const f32x4 &v, float inv, const f32x4 &scale) {
    return pack4(f32x4{v[0] * inv * scale[0], v[1] * inv * scale[1], v[2] * inv * scale[2], v[3] * inv * scale[3]});
}
// cuda/ops.cuh:68-80: the rounded input gradient; the token's g * z terms of the scale gradient go to gz
TG_DEVICE f32x4 normalize_backward(const f32x4 &v, float inv, const f32x4 &g, const f32x4 &scale, float *gz, const Lane &p) {
    f32x4 z, dz, dx;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        z[i] = v[i] * inv;
        dz[i] = g[i] * scale[i];
        gz[4 * i] = g[i] * z[i];
    }
    const float dot = token_dot(dz, z, p);
#pragma unroll
    for (int i = 0; i < 4; ++i)
        dx[i] = round_bf16((dz[i] - z[i] * dot * (1.f / 16.f)) * inv);
    return dx;
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

// ---- teams -------------------------------------------------------------------------------------------
// A team's waves each hold the lanes of all its tokens.  Role 0 has what is one chain - norms, projections of sixteen outputs,
// attention, residuals - and roles 1 to 3 sixteen of the 48 features of the MLP each, forward and backward; the head's 256 logits
// are shared by all four.  A sum over features or logits is still one wave's chain of fmaf in their order, so a
// result does not depend on the roles.  What one wave's work another needs goes through LDS, a tile at a time.
// A lone wave (R = 1) has all of it.
struct Exchange {
    unsigned char *at, *quarters;
    int lane, c;
    TG_DEVICE Exchange(const Model &m, unsigned char *memory, const Lane &p, bool rows)
        : at(memory + teams_at(m.depth, m.teams) + p.team * team_bytes(m.depth, rows)), quarters(memory + embedding_at(m.depth) + p.team * 4096),
          lane(p.lane), c(p.c) {}
    // the input of the MLP or of the head; the place of the last tile
    TG_DEVICE u32x2 &row() const { return reinterpret_cast<u32x2 *>(at + 15 * 1024)[lane]; }
    // activation; or the gradients of gate and up, and behind them the gradient that they come from; or the logits' gradients.  In
    // 32 bits, so that who waits for them need not take them apart.
    TG_DEVICE f32x4 &tile(int k) const { return reinterpret_cast<f32x4 *>(at)[k * 64 + lane]; }
    TG_DEVICE float &high(int role) const { return reinterpret_cast<float *>(at + 16 * 1024)[role * W + c]; }
    TG_DEVICE float &picked(int role) const { return reinterpret_cast<float *>(at + 16 * 1024 + ROLES * W * 4)[role * W + c]; }
    TG_DEVICE f32x4 &quarter(int role) const { return reinterpret_cast<f32x4 *>(quarters)[role * 64 + lane]; }
};
// What the block's waves have written to LDS is there for all of them.  Each role comes here as often as the others.
TG_DEVICE void meet() {
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}
// The rows of a layer that the backward pass wants: in the team's LDS, or in memory.
template <bool LDS> struct Rows {
    unsigned char *at;
    int64_t apart; // from one layer to the next
    int lane, c;
    TG_DEVICE Rows(const Model &m, unsigned char *memory, const Workspace &s, const Lane &p) : lane(p.lane), c(p.c) {
        if constexpr (LDS)
            at = memory + teams_at(m.depth, m.teams) + p.team * team_bytes(m.depth, true) + EXCHANGE_BYTES, apart = ROW_BYTES;
        else
            at = s.rows + size_t(p.wave) * LONE_ROW_BYTES, apart = int64_t(s.waves) * LONE_ROW_BYTES;
    }
    TG_DEVICE u32x2 &tile(int l, int k) const { return reinterpret_cast<u32x2 *>(at + l * apart)[k * 64 + lane]; }
    TG_DEVICE u32x2 &features(int l, int k) const { return reinterpret_cast<u32x2 *>(at + l * apart + ROW_FEATURES)[k * 64 + lane]; }
    TG_DEVICE float &word(int l, int k) const { return reinterpret_cast<float *>(at + l * apart + ROW_TILES * 512)[k * 64 + lane]; }
    TG_DEVICE uint8_t &distance(int l) const { return (at + l * apart + ROW_DISTANCE)[lane]; }
    TG_DEVICE float &inverse(int l, int k) const { return reinterpret_cast<float *>(at + l * apart + ROW_INVERSE)[k * W + c]; }
};
// A layer's, as they are wanted
template <int R> struct LayerRows {
    u32x2 x, query, key, value, middle, features[R == 1 ? 6 : 1];
    float gate, slope, inv1, inv2;
    int distance;
    template <class Rows> TG_DEVICE void request(const Rows &rows, int l) {
        if constexpr (R == 1)
#pragma unroll
            for (int k = 0; k < 6; ++k)
                features[k] = rows.features(l, k);
        x = rows.tile(l, R_X), query = rows.tile(l, R_Q), key = rows.tile(l, R_KEY), value = rows.tile(l, R_VALUE);
        middle = rows.tile(l, R_MIDDLE), gate = rows.word(l, R_GATE), slope = rows.word(l, R_SLOPE);
        inv1 = rows.inverse(l, 0), inv2 = rows.inverse(l, 1), distance = rows.distance(l);
    }
};
// A row for the launch of the weight gradients, written through to memory: what the L2s hold of a launch's results is written back
// behind its last block, and this one leaves 28 MB of such rows at depth 4, 10240 tokens (63.0 us a step, 59.8 so).
TG_DEVICE void leave(u32x2 &to, const u32x2 &v) {
    __hip_atomic_store(reinterpret_cast<uint64_t *>(&to), __builtin_bit_cast(uint64_t, v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
TG_DEVICE u32x2 *operands_of(const Workspace &s, const Lane &p, int l) {
    return s.tiles + (size_t(l) * s.waves + p.wave) * OPERANDS * 64 + p.lane;
}

// ---- forward ---------------------------------------------------------------------------------------
// What role 0 keeps of the head for the backward pass.
struct Head {
    u32x2 hidden;
    float inverse;
};
TG_DEVICE f32x4 embedding_row(const Model &m, const unsigned char *memory, const Lane &p, int token) {
    const bf16_t *row = reinterpret_cast<const bf16_t *>(memory + embedding_at(m.depth)) + token * W + p.g;
    return p.live ? f32x4{bf16_to_float(row[0]), bf16_to_float(row[4]), bf16_to_float(row[8]), bf16_to_float(row[12])} : ZERO;
}
// Sixteen features of the packed gate|up projection and of SwiGLU (cuda/model.cuh:22-29, cuda/ops.cuh:120-131: RN after SiLU and after
// the product).  Roles 1 to 3 keep gate, up and the sigmoid of a layer in registers for the backward pass.
struct Features {
    u32x2 gate, up;
    f32x4 sigmoid;
    TG_DEVICE u32x2 activation() const { return pack4(rounded(unpack4(gate) * sigmoid) * unpack4(up)); }
};
TG_DEVICE f32x4 sigmoids(const u32x2 &gate) {
    f32x4 v = unpack4(gate);
#pragma unroll
    for (int r = 0; r < 4; ++r)
        v[r] = sigmoid(v[r]);
    return v;
}
struct GateUp {
    f32x4 of_both[2];
    TG_DEVICE GateUp(const Staged &weight, int l, int t) : of_both{weight(l * LAYER_TILES + 4 + t), weight(l * LAYER_TILES + 7 + t)} {}
    TG_DEVICE Features operator()(const f32x4 &row) {
        f32x4 both[2];
        multiply_all(of_both, row, both);
        const u32x2 gate = pack4(both[0]);
        return {gate, pack4(both[1]), sigmoids(gate)};
    }
};
// Down projection and SwiGLU backward (cuda/model.cuh:72-80, cuda/ops.cuh:133-144) of sixteen features: what does not wait for the
// gradient, and the gradients of gate and up
struct FeaturesBackward {
    f32x4 down, up, sig, silu, slope;
    TG_DEVICE FeaturesBackward(const Staged &weight, int l, int t, const Features &f)
        : down(weight.turned_feed(l * LAYER_TILES + 10 + t)), up(unpack4(f.up)), sig(f.sigmoid) {
        const f32x4 gate = unpack4(f.gate);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            silu[r] = gate[r] * sig[r];
            slope[r] = fmaf(gate[r], 1.f - sig[r], 1.f);
        }
        silu = rounded(silu);
    }
    TG_DEVICE void operator()(const f32x4 &dh, u32x2 &dgate, u32x2 &dup) const {
        const f32x4 dy = rounded(multiply(down, dh)), da = rounded(dy * up);
        dgate = pack4(da * sig * slope), dup = pack4(dy * silu);
    }
};
// The layers, role 0 (cuda/model.cuh:8-31).  GRADIENT: rows are kept.  h: the embedding's rows, and then the last layer's.
template <int R, bool GRADIENT, int CONTEXT, class Rows>
TG_DEVICE void forward_chain(const Model &m, const Lane &p, const Staged &weight, const Exchange &x, const Rows &rows, const Workspace &s,
                             f32x4 &h, float rc, float rs) {
    const int context = CONTEXT ? CONTEXT : m.context;
    for (int l = 0; l < m.depth; ++l) {
        const int tile = l * LAYER_TILES;
        // QKV projection, RoPE (cuda/model.cuh:14-19)
        f32x4 of_qkv[3] = {weight(tile), weight(tile + 1), weight(tile + 2)};
        const float inv1 = inverse_rms(h, p);
        const u32x2 n1 = normalize(h, inv1, weight.scale(2 * l));
        f32x4 qkv[3];
        multiply_all(of_qkv, unpack4(n1), qkv);
        const f32x4 query = rounded(rotate(rounded(qkv[0]), rc, rs));
        const u32x2 key = pack4(rotate(rounded(qkv[1]), rc, rs));
        const u32x2 value = pack4(qkv[2]);
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
        const f32x4 a = turned(rounded(unpack4(best_value) * gate));
        // output projection and residual: a bf16 add (cuda/model.cuh:20-21, cuda/mma.cuh:95-97)
        const f32x4 middle = rounded(rounded(multiply(weight(tile + 3), a)) + h);
        const float inv2 = inverse_rms(middle, p);
        const u32x2 n2 = normalize(middle, inv2, weight.scale(2 * l + 1));
        u32x2 *operand = operands_of(s, p, l);
        const auto keep = [&] {
            if constexpr (GRADIENT) {
                rows.tile(l, R_X) = pack4(h);
                rows.tile(l, R_Q) = pack4(query);
                rows.tile(l, R_KEY) = best_key;
                rows.tile(l, R_VALUE) = best_value;
                rows.tile(l, R_MIDDLE) = pack4(middle);
                rows.word(l, R_GATE) = gate;
                rows.word(l, R_SLOPE) = fmaf(top * 0.3989422804014327f, expf(-0.5f * top * top), 0.5f * e);
                rows.distance(l) = uint8_t(distance);
                rows.inverse(l, 0) = inv1, rows.inverse(l, 1) = inv2;
                leave(operand[T_N1 * 64], n1);
                leave(operand[T_A * 64], pack4(a));
                leave(operand[T_N2 * 64], n2);
            }
        };
        f32x4 act[3], down[3];
        if constexpr (R == 1) {
            keep();
#pragma unroll
            for (int t = 0; t < 3; ++t) {
                const Features f = GateUp(weight, l, t)(unpack4(n2));
                const u32x2 act_row = f.activation();
                act[t] = unpack4(act_row), down[t] = weight(tile + 10 + t);
                if constexpr (GRADIENT) {
                    rows.features(l, t) = f.gate, rows.features(l, 3 + t) = f.up;
                    leave(operand[(T_ACT + t) * 64], act_row);
                }
            }
        } else {
            x.row() = n2;
            meet(); // the MLP's features are worked on
#pragma unroll
            for (int t = 0; t < 3; ++t)
                down[t] = weight(tile + 10 + t);
            keep();
            ready(down[0], down[1], down[2]);
            meet();
#pragma unroll
            for (int t = 0; t < 3; ++t)
                act[t] = x.tile(t);
        }
        // down projection and residual (cuda/model.cuh:30)
        f32x4 out = ZERO;
#pragma unroll
        for (int t = 0; t < 3; ++t)
            out = multiply(down[t], act[t], out);
        h = rounded(rounded(out) + middle);
    }
}
template <bool GRADIENT>
TG_DEVICE void forward_features(const Model &m, const Lane &p, const Staged &weight, const Exchange &x, const Workspace &s,
                                Features (&kept)[MAX_DEPTH]) {
    const int t = p.role - 1;
    u32x2 *operand = operands_of(s, p, 0) + (T_ACT + t) * 64;
#pragma unroll
    for (int l = 0; l < MAX_DEPTH; ++l) {
        if (l >= m.depth)
            break;
        GateUp project(weight, l, t);
        ready(project.of_both[0], project.of_both[1]);
        meet();
        kept[l] = project(unpack4(x.row()));
        const u32x2 act_row = kept[l].activation();
        x.tile(t) = unpack4(act_row);
        meet();
        if constexpr (GRADIENT)
            leave(operand[size_t(l) * s.waves * (OPERANDS * 64)], act_row);
    }
}
// cuda/model.cuh:8-59, all roles.  dlogits = RN_bf16((p - onehot) / tokens), left in memory and in LDS or, by a lone wave, in `head`.
template <int R> struct Kept {
    Features of_role[MAX_DEPTH];
};
template <> struct Kept<1> {
    u32x2 dlogits[HEAD_TILES];
};
template <int R, bool GRADIENT, int CONTEXT, class Rows>
TG_DEVICE void forward_pass(const Model &m, const Lane &p, const Staged &weight, const Exchange &x, const Rows &rows, const Workspace &s,
                            f32x4 h, int target, float rc, float rs, float *__restrict__ token_losses, float *__restrict__ logits_out,
                            Head &head, Kept<R> &kept) {
    constexpr int TILES = HEAD_TILES / R;
    u32x2 nf;
    if (R == 1 || p.role == 0) {
        forward_chain<R, GRADIENT, CONTEXT>(m, p, weight, x, rows, s, h, rc, rs);
        // final RMSNorm (cuda/model.cuh:32-34)
        const float inv = inverse_rms(h, p);
        nf = normalize(h, inv, weight.scale(2 * m.depth));
        if constexpr (R > 1)
            x.row() = nf;
        if constexpr (GRADIENT) {
            head.hidden = pack4(h), head.inverse = inv;
            s.nf[size_t(p.wave) * 64 + p.lane] = nf;
        }
    } else if constexpr (R > 1)
        forward_features<GRADIENT>(m, p, weight, x, s, kept.of_role);
    // head, softmax cross-entropy (cuda/model.cuh:35-58): this role's tile i is the head's tile role + R i, whose register r is
    // logit 16 (role + R i) + 4 r + g
    f32x4 logit[TILES];
    if constexpr (R > 1) {
        f32x4 of_head[TILES];
#pragma unroll
        for (int i = 0; i < TILES; ++i)
            of_head[i] = weight(weight.head + p.role + R * i), ready(of_head[i]);
        meet();
        multiply_all(of_head, unpack4(x.row()), logit);
    } else
#pragma unroll
        for (int i = 0; i < TILES; ++i)
            logit[i] = multiply(weight(weight.head + i), unpack4(nf));
    float high = -INFINITY;
#pragma unroll
    for (int i = 0; i < TILES; ++i) {
        logit[i] = rounded(logit[i]);
        high = fmaxf(fmaxf(high, fmaxf(logit[i][0], logit[i][1])), fmaxf(logit[i][2], logit[i][3]));
    }
    high = token_max(high);
    if constexpr (R > 1) {
        x.high(p.role) = high;
        meet();
        high = fmaxf(fmaxf(x.high(0), x.high(1)), fmaxf(x.high(2), x.high(3)));
    }
    if (logits_out && p.live)
#pragma unroll
        for (int i = 0; i < TILES; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                logits_out[size_t(p.token) * V + (p.role + R * i) * 16 + 4 * r + p.g] = logit[i][r];
    // the target's logit: register target / 4 % 4 of tile target / 16, of the lane g = target % 4
    const bool holder = p.g == (target & 3) && p.role == (target >> 4) % R;
    const int tile = (target >> 4) / R, mine = holder ? tile * 4 + ((target >> 2) & 3) : -1; // 4 i + r
    float picked = 0.f;
    if constexpr (R == 1) { // by halves: one after another the 64 choices made lone waves spill 8 to 15 registers
        float of_four[TILES];
#pragma unroll
        for (int i = 0; i < TILES; ++i) {
            const float even = target & 4 ? logit[i][1] : logit[i][0], odd = target & 4 ? logit[i][3] : logit[i][2];
            of_four[i] = target & 8 ? odd : even;
        }
#pragma unroll
        for (int half = TILES / 2, bit = 1; half; half >>= 1, bit <<= 1)
#pragma unroll
            for (int i = 0; i < half; ++i)
                of_four[i] = tile & bit ? of_four[2 * i + 1] : of_four[2 * i];
        picked = holder ? of_four[0] : 0.f;
    }
#pragma unroll
    for (int i = 0; i < TILES; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            if constexpr (R > 1)
                picked = 4 * i + r == mine ? logit[i][r] : picked;
            logit[i][r] = expf(logit[i][r] - high);
        }
    picked = swap_add_16(swap_add_32(picked));
    // the sum's tree: every 64th logit in order, then halves of what is left (bits 5 .. 0 of the logit's number)
    f32x4 quarter[4];
    if constexpr (R > 1) {
        x.quarter(p.role) = ((logit[0] + logit[1]) + logit[2]) + logit[3];
        x.picked(p.role) = picked;
        meet();
#pragma unroll
        for (int q = 0; q < 4; ++q)
            quarter[q] = x.quarter(q);
        picked = ((x.picked(0) + x.picked(1)) + x.picked(2)) + x.picked(3);
    } else
#pragma unroll
        for (int q = 0; q < 4; ++q)
            quarter[q] = ((logit[q] + logit[q + 4]) + logit[q + 8]) + logit[q + 12];
    const f32x4 sixteenth = (quarter[0] + quarter[2]) + (quarter[1] + quarter[3]);
    const float sum = swap_add_16(swap_add_32((sixteenth[0] + sixteenth[2]) + (sixteenth[1] + sixteenth[3])));
    if (p.role == 0 && p.live && p.g == 0)
        token_losses[p.token] = high + logf(sum) - picked;
    if constexpr (GRADIENT) {
        const float share = reciprocal(sum), tokens = float(m.tokens), per_token = 1.f / tokens;
#pragma unroll
        for (int i = 0; i < TILES; ++i) {
            f32x4 d;
#pragma unroll
            for (int r = 0; r < 4; ++r)
                d[r] = divide(divide(logit[i][r], sum, share) - (4 * i + r == mine ? 1.f : 0.f), tokens, per_token);
            u32x2 packed = pack4(d);
            packed.x = p.live ? packed.x : 0, packed.y = p.live ? packed.y : 0;
            if constexpr (R > 1)
                x.tile(p.role + R * i) = unpack4(packed);
            else
                kept.dlogits[i] = packed;
            leave(s.dlogits[(size_t(p.wave) * 16 + p.role + R * i) * 64 + p.lane], packed);
        }
    }
}

// ---- backward --------------------------------------------------------------------------------------
// cuda/model.cuh:61-99, without the weight gradients.  Role 0:
template <int R, int CONTEXT, class Rows>
TG_DEVICE void backward_chain(const Model &m, const Lane &p, const Staged &weight, const Exchange &x, const Rows &rows, const Workspace &s,
                              float rc, float rs, const Head &head, const Kept<R> &kept) {
    const int context = CONTEXT ? CONTEXT : m.context;
    auto gz = [&](int norm) { return s.gz + ((size_t(norm) * s.waves + p.wave) * 16 + p.c) * W + p.g; };

    // head input gradient and final RMSNorm backward (cuda/model.cuh:63-66)
    f32x4 dn = ZERO;
    LayerRows<R> next; // a lone wave's are requested while the layer above is worked on
    if constexpr (R == 1) {
        next.request(rows, m.depth - 1);
#pragma unroll
        for (int t = 0; t < 16; ++t)
            dn = multiply(weight.turned_feed(weight.head + t), unpack4(kept.dlogits[t]), dn);
    } else {
        u32x2 of_head[16];
        f32x4 dlogits[16];
#pragma unroll
        for (int t = 0; t < 16; ++t)
            of_head[t] = weight.turned_feed_row(weight.head + t), dlogits[t] = x.tile(t);
        __builtin_amdgcn_sched_barrier(0); // every read goes out before the first product
#pragma unroll
        for (int t = 0; t < 16; ++t)
            dn = multiply(unpack4(of_head[t]), dlogits[t], dn);
    }
    f32x4 dh = normalize_backward(unpack4(head.hidden), head.inverse, rounded(dn), weight.scale(2 * m.depth), gz(2 * m.depth), p);
    for (int l = m.depth - 1; l >= 0; --l) {
        const int tile = l * LAYER_TILES;
        u32x2 *operand = operands_of(s, p, l);
        LayerRows<R> of;
        // down projection, SwiGLU, packed gate|up projection and RMSNorm backward (cuda/model.cuh:72-88)
        if constexpr (R == 1) {
            of = next;
            if (l)
                next.request(rows, l - 1);
            leave(operand[T_DH_DOWN * 64], pack4(dh));
            u32x2 gradient[6];
#pragma unroll
            for (int t = 0; t < 3; ++t) {
                FeaturesBackward(weight, l, t, {of.features[t], of.features[3 + t], sigmoids(of.features[t])})(dh, gradient[t], gradient[3 + t]);
                leave(operand[(T_DGU + t) * 64], gradient[t]);
                leave(operand[(T_DGU + 3 + t) * 64], gradient[3 + t]);
            }
            dn = ZERO;
#pragma unroll
            for (int t = 0; t < 6; ++t)
                dn = multiply(weight.turned_feed(tile + 4 + t), unpack4(gradient[t]), dn);
        } else {
            x.tile(6) = dh;
            meet();
            leave(operand[T_DH_DOWN * 64], pack4(dh));
            f32x4 gate_up[6];
#pragma unroll
            for (int t = 0; t < 6; ++t)
                gate_up[t] = weight.turned_feed(tile + 4 + t);
            of.request(rows, l);
            ready(gate_up[0], gate_up[1], gate_up[2], gate_up[3], gate_up[4], gate_up[5]);
            meet();
            dn = ZERO;
#pragma unroll
            for (int t = 0; t < 6; ++t)
                dn = multiply(gate_up[t], x.tile(t), dn);
        }
        const f32x4 key = unpack4(of.key), value = unpack4(of.value);
        const u32x2 query = of.query;
        const float gate = of.gate;
        // residual gradients stay bf16 between operators (cuda/ops.cuh:74-76)
        dh = rounded(dh + normalize_backward(unpack4(of.middle), of.inv2, rounded(dn), weight.scale(2 * l + 1), gz(2 * l + 1), p));
        leave(operand[T_DH_ATTENTION * 64], pack4(dh));

        // attention: output projection backward, the score gradient of the cached winner, query / key / value gradients
        // gathered over the sequence, inverse RoPE, QKV projection and RMSNorm backward (cuda/model.cuh:89-96,
        // cuda/attention.cuh:72-106)
        const u32x2 dattn = pack4(multiply(weight(weight.turned_attention + l), dh));
        const f32x4 da = unpack4(dattn);
        float dt = 0.f;
#pragma unroll
        for (int c = 0; c < 4; ++c)
            dt = fmaf(da[c], value[c], dt);
        dt *= of.slope;
        f32x4 dk = ZERO, dv = ZERO;
        up_to<0, CONTEXT ? CONTEXT - 1 : 7>([&](auto step) { // queries of this token's sequence that chose it, in order
            constexpr int D = decltype(step)::value;
            if (D >= context)
                return;
            // every lane takes part in the shifts, so none of them may sit behind a condition
            const uint32_t theirs = later<D>(uint32_t(of.distance));
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
        const f32x4 dq = turned(rounded(rotate_back(rounded(key * dt), rc, rs)));
        dk = turned(rounded(rotate_back(rounded(dk), rc, rs)));
        dv = turned(rounded(dv));
        leave(operand[T_DQKV * 64], pack4(dq));
        leave(operand[(T_DQKV + 1) * 64], pack4(dk));
        leave(operand[(T_DQKV + 2) * 64], pack4(dv));
        dn = multiply(weight.turned_natural(tile + 2), dv,
                      multiply(weight.turned_natural(tile + 1), dk, multiply(weight.turned_natural(tile), dq)));
        dh = rounded(dh + normalize_backward(unpack4(of.x), of.inv1, rounded(dn), weight.scale(2 * l), gz(2 * l), p));
    }
    s.dh[size_t(p.wave) * 64 + p.lane] = pack4(dh);
}
TG_DEVICE void backward_features(const Model &m, const Lane &p, const Staged &weight, const Exchange &x, const Workspace &s,
                                 const Features (&kept)[MAX_DEPTH]) {
    const int t = p.role - 1;
#pragma unroll
    for (int l = MAX_DEPTH - 1; l >= 0; --l) {
        if (l >= m.depth)
            continue;
        FeaturesBackward backward(weight, l, t, kept[l]);
        ready(backward.down, backward.up, backward.silu, backward.slope);
        u32x2 dgate, dup;
        meet();
        backward(x.tile(6), dgate, dup);
        x.tile(t) = unpack4(dgate);
        x.tile(3 + t) = unpack4(dup);
        meet();
        u32x2 *operand = operands_of(s, p, l);
        leave(operand[(T_DGU + t) * 64], dgate);
        leave(operand[(T_DGU + 3 + t) * 64], dup);
    }
}
template <int R, int CONTEXT, class Rows>
TG_DEVICE void backward_pass(const Model &m, const Lane &p, const Staged &weight, const Exchange &x, const Rows &rows, const Workspace &s,
                             float rc, float rs, const Head &head, const Kept<R> &kept) {
    if constexpr (R > 1)
        meet(); // the logits' gradients
    if (R == 1 || p.role == 0)
        backward_chain<R, CONTEXT>(m, p, weight, x, rows, s, rc, rs, head, kept);
    else if constexpr (R > 1)
        backward_features(m, p, weight, x, s, kept.of_role);
}

// ---- kernels -----------------------------------------------------------------------------------------
// Four waves a SIMD: of lone waves two blocks share a unit (128 registers; with 155 to 177 and one block 131072 tokens at depth 8 173 us
// forward and 242 with gradient, so 156 and 221; 160 and 230 while 8 to 15 registers were spilled, which cost 524288 tokens at depth 1 372 and
// 444 us for 324 and 387).
template <bool GRADIENT, int R>
__global__ __launch_bounds__(64 * block_waves(R), 4) void w16_forward_kernel(Model m, const uint8_t *__restrict__ x, const uint8_t *__restrict__ y,
                                                                         Workspace s, float *__restrict__ token_losses,
                                                                         float *__restrict__ logits_out) {
    extern __shared__ __align__(16) unsigned char memory[];
    const Lane p = lane_of<R>(m, s.waves);
    const Staged weight(m, memory, p);
    Staging<R> staging(m, memory);
    const int token = p.live ? x[p.token] : 0, target = p.live ? y[p.token] : 0;
    staging.request();
    staging.request_embedding(!(reinterpret_cast<uintptr_t>(m.hi) & 15));
    staging.finish(false);
    if (!staging.stays())
        return;
    const f32x4 h = embedding_row(m, memory, p, token);
    float rc, rs;
    rotation(p.position, rc, rs);
    Head head;
    Kept<R> kept;
    forward_pass<R, GRADIENT, 0>(m, p, weight, Exchange(m, memory, p, false), Rows<false>(m, memory, s, p), s, h, target, rc, rs, token_losses,
                                 logits_out, head, kept);
    if constexpr (GRADIENT)
        if (p.role == 0) {
            const size_t here = size_t(p.wave) * 64 + p.lane;
            s.hidden[here] = head.hidden, s.inverse[here] = head.inverse;
        }
}
template <int R> __global__ __launch_bounds__(64 * block_waves(R)) void w16_backward_kernel(Model m, Workspace s) {
    extern __shared__ __align__(16) unsigned char memory[];
    const Lane p = lane_of<R>(m, s.waves);
    const Staged weight(m, memory, p);
    const Exchange exchange(m, memory, p, false);
    Staging<R> staging(m, memory);
    staging.request();
    const size_t here = size_t(p.wave) * 64 + p.lane;
    const Head head = {s.hidden[here], s.inverse[here]};
    staging.finish(true);
    if (!staging.stays())
        return;
    const Rows<false> rows(m, memory, s, p);
    Kept<R> kept;
#pragma unroll
    for (int i = 0; i < HEAD_TILES / R; ++i) {
        const u32x2 row = s.dlogits[(size_t(p.wave) * 16 + p.role + R * i) * 64 + p.lane];
        if constexpr (R > 1)
            exchange.tile(p.role + R * i) = unpack4(row);
        else
            kept.dlogits[i] = row;
    }
    float rc, rs;
    rotation(p.position, rc, rs);
    if constexpr (R > 1)
        if (p.role)
#pragma unroll
            for (int l = 0; l < MAX_DEPTH; ++l)
                if (l < m.depth)
                    kept.of_role[l] = GateUp(weight, l, p.role - 1)(unpack4(normalize(unpack4(rows.tile(l, R_MIDDLE)), rows.inverse(l, 1), weight.scale(2 * l + 1))));
    backward_pass<R, 0>(m, p, weight, exchange, rows, s, rc, rs, head, kept);
}
// A training step's both passes: a team's backward pass reads only what its own forward pass kept, so the two are one launch
// and the weights are staged once.  us a launch, all on lone waves and so: depth 4, 2560 sequences of 4 38.6 and 31.5; depth 8, four
// batches of 16 of 8 64 and 41.  Of the 31.5 the weights take 2, a layer 2.5 forward and 2.6 back, the head 5.5.  Tokens and targets come straight out of the training
// bytes, every sequence a window at a hashed place (cuda/dataset.cuh:13-27); the tokens are left for the embedding's gradient.
template <int CONTEXT, int R, bool ROWS>
__global__ __launch_bounds__(64 * block_waves(R)) void w16_step_kernel(Model m, W16Data data, uint64_t inverse, Workspace first, Group group) {
    extern __shared__ __align__(16) unsigned char memory[];
    const W16Batch &batch = group.member[blockIdx.y];
    const Workspace s = group.workspace(first, blockIdx.y);
    m.hi = batch.weights.hi, m.lo = batch.weights.lo;
    const Lane p = lane_of<R>(m, s.waves);
    const Staged weight(m, memory, p);
    Staging<R> staging(m, memory);
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
    staging.request();
    staging.request_embedding();
    float rc, rs;
    rotation(p.position, rc, rs);
    ready(rc, rs);
    staging.finish(true);
    if (!staging.stays())
        return;
    if (p.live && p.g == 0 && p.role == 0)
        batch.tokens[p.token] = uint8_t(token);
    const f32x4 h = embedding_row(m, memory, p, token);
    const Exchange exchange(m, memory, p, ROWS);
    const Rows<ROWS> rows(m, memory, s, p);
    Head head;
    Kept<R> kept;
    forward_pass<R, true, CONTEXT>(m, p, weight, exchange, rows, s, h, target, rc, rs, batch.token_losses, nullptr, head, kept);
    backward_pass<R, CONTEXT>(m, p, weight, exchange, rows, s, rc, rs, head, kept);
}

// ---- weight gradients ------------------------------------------------------------------------------
// A block sums what one layer (or the head, or the embedding) has of a chunk's tokens, in token order: partial[chunk].  Its
// rows come to LDS as the waves kept them; the transposing load then gives lane 16 q + i feature 4 (i % 4) + i / 4 of tokens
// 4 j + q, an operand of the fp32 instruction whose steps run over the tokens.  That moves data and computes nothing: an
// infinity stays in its own feature.  A wave has three or four tiles of the gradient at a time, whose chains of dependent
// instructions fill the matrix pipe, which bounds the kernel together with what the rows take on their way (a team's are
// worked on while the next ones' come): 93 tiles of 32 instructions a chunk at depth 4, and 28 MB of rows.  2560 sequences of 4 there: 15.3 us
// with a wave for each tile that loaded its rows and turned them with the identity matrix, 13.1 with every half of a chunk waited
// for, 12.5 so; four batches of 16 of 8 at depth 8 11.1 and 10.2.
// Half a chunk, as the last one or the only one may be, is all that is worked on: 16 sequences of 4 at depth 4 6.4 us with the
// missing half as zeros, 4.6 so.
constexpr int HEAD_ROWS = 17; // the head's tiles of a wave in LDS: dlogits, and the normalised rows
constexpr size_t GRADIENT_LDS = size_t(CHUNK_WAVES) * OPERANDS * 512;
static_assert(HEAD_ROWS <= OPERANDS, "the head's rows fit a layer's");
// a lane's rows 4 r + g and column 4 (c % 4) + c / 4 of a gradient tile
TG_DEVICE void store_tile(float *out, const f32x4 &sum, int width, int lane) {
    const int g = lane >> 4, column = feed_row(lane & 15);
#pragma unroll
    for (int r = 0; r < 4; ++r)
        out[(4 * r + g) * width + column] = sum[r];
}
// the g * z terms of a norm's scale: token 4 j + g of every wave, feature c
struct ScaleTerms {
    float v[CHUNK_WAVES][4];
    TG_DEVICE void request(const Workspace &s, int norm, int first, int waves, int lane) {
        const float *gz = s.gz + (size_t(norm) * s.waves + first) * 16 * W + lane;
#pragma unroll
        for (int w = 0; w < CHUNK_WAVES; ++w)
#pragma unroll
            for (int j = 0; j < 4; ++j)
                v[w][j] = w < waves ? gz[(w * 4 + j) * 64] : 0.f;
    }
    // a row of ones times the terms; lane c of the first sixteen has feature c
    TG_DEVICE float sum() const {
        f32x4 scale = ZERO;
#pragma unroll
        for (int w = 0; w < CHUNK_WAVES; ++w)
#pragma unroll
            for (int j = 0; j < 4; ++j)
                scale = __builtin_amdgcn_mfma_f32_16x16x4f32(1.f, v[w][j], scale, 0, 0, 0);
        return scale[0];
    }
};
// TILES chains of products over the tokens of one team.  `rows` and `columns`: this lane's place in the team's tiles.
template <int TILES>
TG_DEVICE void add_team(f32x4 (&sum)[4], const unsigned char *const (&rows)[TILES], const unsigned char *const (&columns)[TILES]) {
    f32x4 a[TILES], b[TILES];
#pragma unroll
    for (int n = 0; n < TILES; ++n)
        a[n] = unpack4(read_across(rows[n])), b[n] = unpack4(read_across(columns[n]));
#pragma unroll
    for (int n = 0; n < TILES; ++n)
        ready(a[n], b[n]);
    products_only();
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int n = 0; n < TILES; ++n)
            sum[n] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[n][j], b[n][j], sum[n], 0, 0, 0);
    products_only();
}
__global__ __launch_bounds__(64 * WAVES) void w16_weight_gradient_kernel(Model m, Workspace whole, Group group, int parameters) {
    extern __shared__ __align__(16) unsigned char memory[];
    const Workspace s = group.workspace(whole, blockIdx.y);
    const uint8_t *x = group.member[blockIdx.y].tokens;
    // consecutive blocks sit on consecutive XCDs: block 8 i + k takes the i-th unit of XCD k's chunks
    const int units = m.depth + 2, chunk = (blockIdx.x >> 3) / units * 8 + (blockIdx.x & 7), unit = (blockIdx.x >> 3) % units;
    if (chunk >= s.chunks)
        return;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), c = lane & 15, g = lane >> 4;
    const int first = chunk * CHUNK_WAVES, waves = min(CHUNK_WAVES, s.waves - first);
    const bool second_half = waves > CHUNK_WAVES / 2;
    float *out = s.partials + size_t(chunk) * parameters;
    const uint32_t lds = lds_address(memory);
    // `tiles` tiles of every team, which lie one behind another in memory and do in LDS; 16 bytes a lane.  The last chunk's missing
    // teams are zeros, of the second half only where it has any.
    const auto copy = [&](auto tiles, const u32x2 *source, int to) {
        constexpr int COPIES = decltype(tiles)::value;
        static_assert(CHUNK_WAVES * 512 == 64 * WAVES * 16, "every wave has a copy for each of a team's tiles");
        const unsigned char *from = reinterpret_cast<const unsigned char *>(uniform(source)) + wave * 1024;
        const uint32_t at = lds + uint32_t(to + wave * 1024);
        if (waves == CHUNK_WAVES) {
#pragma unroll
            for (int i = 0; i < COPIES; ++i)
                async_copy16(at + uint32_t(i) * WAVES * 1024, from + i * WAVES * 1024, uint32_t(lane * 16));
            return;
        }
        const int there = waves * COPIES * 512, wanted = (second_half ? CHUNK_WAVES : CHUNK_WAVES / 2) * COPIES * 512;
        for (int i = 0; i < COPIES; ++i) {
            const int piece = (i * WAVES + wave) * 1024 + lane * 16;
            if (piece < there)
                async_copy16(at + uint32_t(i) * WAVES * 1024, from + i * WAVES * 1024, uint32_t(lane * 16));
            else if (piece < wanted)
                *reinterpret_cast<u32x4 *>(memory + to + piece) = u32x4{0, 0, 0, 0};
        }
    };
    // The teams' rows one after another, each as soon as it is there: team w's last tile is brought by a wave's copy
    // ceil((w + 1) tiles / 8) - 1 of `tiles`.  A chunk that is not full has fewer copies: all of them are waited for.
    // The wave's loads behind its copies, `younger` of them, may stay under way.
    const auto each_team = [&](auto tiles, auto younger, auto &&add) {
        constexpr int COPIES = decltype(tiles)::value, YOUNGER = decltype(younger)::value;
        up_to<0, CHUNK_WAVES - 1>([&](auto team) {
            constexpr int TEAM = decltype(team)::value;
            if (TEAM >= CHUNK_WAVES / 2 && !second_half)
                return;
            if (waves == CHUNK_WAVES)
                wait_vmcnt<COPIES - ((TEAM + 1) * COPIES + CHUNK_WAVES - 1) / CHUNK_WAVES + YOUNGER>();
            else if (TEAM == 0) {
                wait_vmcnt<0>();
                wait_lgkmcnt0();
            }
            if (TEAM == 0 || waves == CHUNK_WAVES)
                __syncthreads();
            add(team);
        });
    };
    const unsigned char *mine = memory + across_offset(lane, true);
    const auto tile = [&](int n) { return mine + n * 512; };
    f32x4 sum[4] = {ZERO, ZERO, ZERO, ZERO};
    ScaleTerms terms;
    if (unit < m.depth) {
        const Layer q = layer_layout(unit);
        copy(std::integral_constant<int, OPERANDS>{}, s.tiles + (size_t(unit) * s.waves + first) * OPERANDS * 64, 0);
        constexpr std::integral_constant<int, OPERANDS> tiles;
        if (wave == 0)
            each_team(tiles, std::integral_constant<int, 0>{}, [&](auto team) {
                const unsigned char *at = tile(decltype(team)::value * OPERANDS), *n1 = at + T_N1 * 512, *dqkv = at + T_DQKV * 512;
                add_team<4>(sum, {dqkv, dqkv + 512, dqkv + 1024, at + T_DH_ATTENTION * 512}, {n1, n1, n1, at + T_A * 512});
            });
        else if (wave == 3)
            each_team(tiles, std::integral_constant<int, 0>{}, [&](auto team) {
                const unsigned char *at = tile(decltype(team)::value * OPERANDS), *dh = at + T_DH_DOWN * 512, *act = at + T_ACT * 512;
                add_team<3>(sum, {dh, dh, dh}, {act, act + 512, act + 1024});
            });
        else { // waves 1 and 2 have a norm's scale besides gate and up
            terms.request(s, 2 * unit + wave - 1, first, waves, lane);
            each_team(tiles, std::integral_constant<int, CHUNK_WAVES * 4>{}, [&](auto team) {
                const unsigned char *at = tile(decltype(team)::value * OPERANDS), *dgu = at + (T_DGU + 3 * wave - 3) * 512, *n2 = at + T_N2 * 512;
                add_team<3>(sum, {dgu, dgu + 512, dgu + 1024}, {n2, n2, n2});
            });
            const float scale = terms.sum();
            if (g == 0)
                out[(wave == 1 ? q.attention_norm : q.mlp_norm) + c] = scale;
        }
        if (wave == 0) {
#pragma unroll
            for (int t = 0; t < 4; ++t) // the attention projection lies behind q, k, v
                store_tile(out + q.qkv + t * 256, sum[t], W, lane);
            return;
        }
#pragma unroll
        for (int t = 0; t < 3; ++t)
            store_tile(wave == 3 ? out + q.down + t * 16 : out + q.gate + ((wave - 1) * 3 + t) * 256, sum[t], wave == 3 ? F : W, lane);
        return;
    }
    if (unit == m.depth) { // the head: a wave four tiles of logits
        constexpr int NF = CHUNK_WAVES * 16;
        copy(std::integral_constant<int, 1>{}, s.nf + size_t(first) * 64, NF * 512);
        copy(std::integral_constant<int, 16>{}, s.dlogits + size_t(first) * 16 * 64, 0);
        const auto add = [&](auto team) {
            constexpr int TEAM = decltype(team)::value;
            const unsigned char *of_wave = tile(TEAM * 16 + wave * 4), *nf = tile(NF + TEAM);
            add_team<4>(sum, {of_wave, of_wave + 512, of_wave + 1024, of_wave + 1536}, {nf, nf, nf, nf});
        };
        const int at = V * W + m.depth * LAYER_SIZE + W;
        if (wave == 0) {
            terms.request(s, 2 * m.depth, first, waves, lane);
            each_team(std::integral_constant<int, 16>{}, std::integral_constant<int, CHUNK_WAVES * 4>{}, add);
            const float scale = terms.sum();
            if (g == 0)
                out[at - W + c] = scale;
        } else
            each_team(std::integral_constant<int, 16>{}, std::integral_constant<int, 0>{}, add);
#pragma unroll
        for (int t = 0; t < 4; ++t)
            store_tile(out + at + (wave * 4 + t) * 256, sum[t], W, lane);
        return;
    }
    // The embedding's rows: the one-hot matrix of the tokens times the gradient.  0 times an infinity is NaN, in ids that have
    // no part in it, so where a row is not finite the rows are added one by one.
    copy(std::integral_constant<int, 1>{}, s.dh + size_t(first) * 64, 0);
    uint32_t ids[CHUNK_WAVES];
#pragma unroll
    for (int w = 0; w < CHUNK_WAVES; ++w) {
        ids[w] = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) // rows beyond the last token are zero: any id will do, and every load goes out at once
            ids[w] |= uint32_t(x[min((first + w) * m.per_wave + min(4 * j + g, m.per_wave - 1), m.tokens - 1)]) << (8 * j);
    }
    wait_vmcnt<0>();
    wait_lgkmcnt0();
    __syncthreads();
    const int vocabulary = wave * 64; // of the four tiles' first id
    bool extreme = false;
#pragma unroll
    for (int w = 0; w < CHUNK_WAVES; ++w) {
        if (w == CHUNK_WAVES / 2 && !second_half)
            break;
        const u32x2 row = read_across(tile(w));
        const auto either = [](uint32_t two) { return (two & 0x7f80u) == 0x7f80u || (two & 0x7f800000u) == 0x7f800000u; };
        extreme = extreme || either(row.x) || either(row.y);
        const f32x4 b = unpack4(row);
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int t = 0; t < 4; ++t)
                sum[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(int((ids[w] >> (8 * j)) & 255u) == vocabulary + t * 16 + c ? 1.f : 0.f, b[j],
                                                              sum[t], 0, 0, 0);
    }
    if (__builtin_amdgcn_ballot_w64(extreme)) {
        sum[0] = sum[1] = sum[2] = sum[3] = ZERO;
#pragma unroll 1
        for (int w = 0; w < waves; ++w)
#pragma unroll 1
            for (int t = 0; t < m.per_wave; ++t) {
                const int token = (first + w) * m.per_wave + t;
                if (token >= m.tokens)
                    break;
                // column 4 (c % 4) + c / 4 is element c % 4 of item (c / 4, t)
                const float value = bf16_to_float(reinterpret_cast<const bf16_t *>(memory)[(w * 64 + 16 * (c >> 2) + t) * 4 + (c & 3)]);
                const int id = int(x[token]) - vocabulary - 4 * g;
#pragma unroll
                for (int n = 0; n < 4; ++n)
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        sum[n][r] = id == 16 * n + r ? sum[n][r] + value : sum[n][r];
            }
    }
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) // the ids are in their own order
            out[(vocabulary + t * 16 + 4 * g + r) * W + feed_row(c)] = sum[t][r];
}
// gradient = the chunks' sums in chunk order, an element a thread, whose loads are in flight together: 80 chunks of 21648
// parameters took 5.9 us with four elements a thread on a quarter of the blocks and sixteen loads at a time, 5.2 so.  Four
// chunks and fewer ask forty times for nothing: 1 chunk 2.5 us, with four at a time 1.2.
// Where norms are wanted, four blocks leave the parts of one sum of squares, of 1024 elements (FOLD_QUARTERS).
// Blocks beyond the parameters average the losses: one a position, in double (cuda/trainer.cuh:79-100).
constexpr int FOLD_QUARTERS = 4;
int fold_blocks(int parameters) { return (parameters + 1023) / 1024 * FOLD_QUARTERS; }
__global__ __launch_bounds__(256) void w16_fold_kernel(Workspace whole, Group group, int parameters, int blocks, int batch,
                                                       int context) {
    const W16Batch &member = group.member[blockIdx.y];
    const float *partials = group.workspace(whole, blockIdx.y).partials;
    const int chunks = whole.chunks;
    if (int(blockIdx.x) >= blocks) {
        __shared__ double sums[4];
        const int position = blockIdx.x - blocks;
        double sum = 0;
#pragma unroll 4
        for (int b = threadIdx.x; b < batch; b += 256)
            sum += member.token_losses[size_t(b) * context + position];
#pragma unroll
        for (int k = 32; k; k >>= 1)
            sum += __shfl_xor(sum, k, 64);
        if ((threadIdx.x & 63) == 0)
            sums[threadIdx.x >> 6] = sum;
        __syncthreads();
        if (threadIdx.x == 0)
            member.means[position] = float(((sums[0] + sums[1]) + (sums[2] + sums[3])) / batch);
        return;
    }
    __shared__ __align__(16) float row[256];
    const int at = blockIdx.x * 256 + threadIdx.x;
    float sum = 0.f;
    if (at < parameters) {
        const float *from = partials + at;
        const auto add = [&](auto at_once) {
            constexpr int AT_ONCE = decltype(at_once)::value;
            for (int c = 0; c < chunks; c += AT_ONCE) {
                float v[AT_ONCE];
#pragma unroll
                for (int i = 0; i < AT_ONCE; ++i)
                    if (c + i < chunks)
                        v[i] = from[size_t(c + i) * parameters];
#pragma unroll
                for (int i = 0; i < AT_ONCE; ++i)
                    if (c + i < chunks)
                        sum += v[i];
            }
        };
        if (chunks <= 4)
            add(std::integral_constant<int, 4>{});
        else
            add(std::integral_constant<int, 40>{});
        member.gradient[at] = sum;
    }
    if (!member.norms)
        return;
    row[threadIdx.x] = sum;
    __syncthreads();
    if (threadIdx.x < 64) {
        const float squares = wave_sum(0.f + quad_squares(reinterpret_cast<const f32x4 *>(row)[threadIdx.x]));
        if (threadIdx.x == 0)
            member.norms[blockIdx.x] = squares;
    }
}

// ---- optimizer (cuda/optim.cuh:17-119) ------------------------------------------------------------------
// Blocks 0 .. 5 depth - 1: Muon, a hidden matrix each.  The rest: AdamW, 256 quads of embedding, scales and head each.
// The Newton-Schulz iterate is a 16 x n matrix in 16 x 16 tiles, one a wave, lane 16 g + c holding rows 4 g .. of column c;
// the products run on the fp32 matrix instruction (the same fmaf chains as a loop).  X X^T is symmetric to the last bit,
// so its tile turned is the operand of the two products behind it, every wave computes it for itself, and a step of the
// iteration exchanges nothing but X through LDS.
// One launch makes as many steps, one after another, as there are gradients at hand: an element's (Muon: a matrix's) weights
// and state stay in the registers between them.  What a matrix's iteration starts from hangs on gradients and momentum alone, so
// up to four steps' iterations run side by side, each on a group of four waves, and only the weights' own chain is left in the steps'
// order: every group follows it and writes its step's.
constexpr int UPDATE_GROUPS = 4;
struct Update {
    float *momentum, *variance;
    int norm_count, norm_parts, depth; // norms: norm_count sums of norm_parts partial sums each, 1 or FOLD_QUARTERS
    int count, ns_steps;
    W16Step step[W16_BATCHES];
};
// Clip factor of step n, by one wave: the sums of a fold's quarters first, then as clip_factor adds them (64 sums at most).
TG_DEVICE float fold_clip(const Update &u, int n, const f32x4 &part) {
    const float sum = int(threadIdx.x & 63) < u.norm_count ? (part[0] + part[1]) + (part[2] + part[3]) : 0.f;
    return fminf(1.f, u.step[n].adam.clip / (sqrtf(wave_sum(0.f + sum)) + 1e-6f));
}
TG_DEVICE f32x4 fold_parts(const Update &u, int n) {
    return int(threadIdx.x & 63) < u.norm_count ? reinterpret_cast<const f32x4 *>(u.step[n].norms)[threadIdx.x & 63] : ZERO;
}
// The clip factors of steps first .. first + groups - 1, for all threads; a group's waves have asked for its `part`.
TG_DEVICE void clip_factors(const Update &u, int first, int groups, const f32x4 &part, float (&clips)[UPDATE_GROUPS], float *waves) {
    const int group = threadIdx.x >> 8;
    if (u.norm_parts == 1) { // more norms than a wave has lanes, in launches of one step
        const float clip = clip_factor(u.step[first].adam.clip, u.step[first].norms, u.norm_count, waves);
        __syncthreads();
        if (threadIdx.x == 0)
            clips[0] = clip;
    } else if ((threadIdx.x & 255) == 0 || u.step[first].adam.clip > 0.f) {
        const float clip = u.step[first].adam.clip > 0.f ? fold_clip(u, min(first + group, u.count - 1), part) : 1.f;
        if ((threadIdx.x & 255) == 0 && group < groups)
            clips[group] = clip;
    }
    __syncthreads();
}
template <int TILES> TG_DEVICE void iterate(u32x2 (&wide)[2][3][64], int steps, int across, int tile, int lane) {
    f32x4 x = unpack4(wide[0][tile][lane]); // rows 4 g .. of column 16 tile + c
    for (int step = 0; step < steps; ++step) {
        const unsigned char *in = reinterpret_cast<const unsigned char *>(wide[step & 1]) + across;
        f32x4 row[TILES], gram = ZERO; // A = X X^T, kept in bf16
#pragma unroll
        for (int k = 0; k < TILES; ++k)
            row[k] = unpack4(read_across(in + k * 512));
#pragma unroll
        for (int k = 0; k < TILES; ++k)
            gram = multiply(row[k], row[k], gram);
        gram = rounded(gram);
        const f32x4 gram_turned = turned(gram), square = multiply(gram_turned, gram_turned);
        f32x4 work; // -4.775 A + 2.0315 A A
#pragma unroll
        for (int r = 0; r < 4; ++r)
            work[r] = fmaf(2.0315f, square[r], -4.775f * gram[r]);
        f32x4 product = multiply(turned(rounded(work)), turned(x));
#pragma unroll
        for (int r = 0; r < 4; ++r)
            product[r] = fmaf(3.4445f, x[r], product[r]);
        const u32x2 packed = pack4(product);
        wide[(step & 1) ^ 1][tile][lane] = packed;
        x = unpack4(packed);
        meet();
    }
}
TG_DEVICE void muon_matrix(const Update &u, int matrix, float (&clips)[UPDATE_GROUPS], float *waves) {
    __shared__ __align__(16) u32x2 wide[UPDATE_GROUPS][2][3][64]; // the iterate's tiles of sixteen columns, as the lanes hold them
    __shared__ float norm_waves[UPDATE_GROUPS][4];
    const Layer p = layer_layout(matrix / 5);
    const int type = matrix % 5;
    const int weight = type == 0 ? p.qkv : type == 1 ? p.attention : type == 2 ? p.gate : type == 3 ? p.up : p.down;
    const int rows = (type == 0 || type == 2 || type == 3) ? 48 : 16, cols = type == 4 ? 48 : 16;
    const int tiles = max(rows, cols) / 16, size = rows * cols, tid = threadIdx.x & 255;
    const int group = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8), groups = blockDim.x >> 8;
    const int lane = tid & 63, tile = __builtin_amdgcn_readfirstlane(tid >> 6), across = across_offset(lane, true);
    // element tid + 256 k of the matrix is this thread's until the iteration and again behind it; its place in the 16 x n form
    float m[3], w[3], g[UPDATE_GROUPS][3];
    int place[3];
    f32x4 part = ZERO;
    const auto request = [&](int first) {
        if (u.norm_parts != 1 && first < u.count)
            part = fold_parts(u, min(first + group, u.count - 1));
#pragma unroll
        for (int n = 0; n < UPDATE_GROUPS; ++n)
            if (n < groups && first + n < u.count)
#pragma unroll
                for (int k = 0; k < 3; ++k)
                    g[n][k] = tid + 256 * k < size ? u.step[first + n].gradient[weight + tid + 256 * k] : 0.f;
    };
    request(0);
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const int i = weight + tid + 256 * k, line = (tid + 256 * k) / cols, at = tid + 256 * k - line * cols;
        const int row = rows > cols ? at : line, col = rows > cols ? line : at;
        place[k] = (((col >> 4) * 64 + (row >> 2) * 16 + (col & 15)) << 2) + (row & 3);
        const bool mine = tid + 256 * k < size;
        m[k] = mine ? u.momentum[i] : 0.f;
        w[k] = mine ? master(u.step[0].from.hi, u.step[0].from.lo, i) : 0.f;
    }
    for (int first = 0; first < u.count; first += groups) {
        const int steps = min(groups, u.count - first);
        clip_factors(u, first, steps, part, clips, waves);
        float squares = 0.f, b[3] = {0.f, 0.f, 0.f};
#pragma unroll
        for (int n = 0; n < UPDATE_GROUPS; ++n) {
            if (n >= steps)
                break;
            const float rate = u.step[first + n].muon.momentum, clip = clips[n];
            float sum = 0.f;
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                const float gs = g[n][k] * clip;
                m[k] = fmaf(1.f - rate, fmaf(g[n][k], clip, -m[k]), m[k]);
                const float mine = round_bf16(fmaf(rate, m[k] - gs, gs));
                if (tid + 256 * k < size)
                    sum = fmaf(mine, mine, sum);
                b[k] = n == group ? mine : b[k];
            }
            squares = n == group ? sum : squares;
        }
        request(first + groups);
        squares = wave_sum(squares);
        if (lane == 0)
            norm_waves[group][tile] = squares;
        __syncthreads();
        const float norm = fmaxf(round_bf16(sqrtf((norm_waves[group][0] + norm_waves[group][1]) + (norm_waves[group][2] + norm_waves[group][3]))),
                                 round_bf16(1e-7f));
#pragma unroll
        for (int k = 0; k < 3; ++k)
            if (tid + 256 * k < size)
                reinterpret_cast<bf16_t *>(wide[group][0])[place[k]] = float_to_bf16(b[k] / norm);
        __syncthreads();
        if (tile >= tiles || group >= steps)
            for (int step = 0; step < u.ns_steps; ++step)
                meet();
        else if (tiles == 3)
            iterate<3>(wide[group], u.ns_steps, across, tile, lane);
        else
            iterate<1>(wide[group], u.ns_steps, across, tile, lane);
#pragma unroll
        for (int n = 0; n < UPDATE_GROUPS; ++n) {
            if (n >= steps)
                break;
            const W16Step &step = u.step[first + n];
            const bf16_t *result = reinterpret_cast<const bf16_t *>(wide[n][u.ns_steps & 1]);
            const float adjusted = step.muon.lr * sqrtf(fmaxf(1.f, float(rows) / float(cols))), keep = fmaf(-step.muon.lr, step.muon.weight_decay, 1.f);
#pragma unroll
            for (int k = 0; k < 3; ++k)
                if (tid + 256 * k < size) {
                    const int i = weight + tid + 256 * k;
                    w[k] = fmaf(w[k], keep, -(adjusted * bf16_to_float(result[place[k]])));
                    if (n == group) {
                        const uint32_t bits = __float_as_uint(w[k]);
                        step.to.hi[i] = uint16_t(bits >> 16); // cuda/ops.cuh:10-14
                        step.to.lo[i] = uint16_t(bits);
                    }
                }
        }
        __syncthreads(); // the next steps' matrices go where these results are read, their clip factors where these are
    }
    if (group == 0)
#pragma unroll
        for (int k = 0; k < 3; ++k)
            if (tid + 256 * k < size)
                u.momentum[weight + tid + 256 * k] = m[k];
}
__global__ __launch_bounds__(256 * UPDATE_GROUPS) void w16_update_kernel(Update u) {
    __shared__ float clips[UPDATE_GROUPS], waves[4];
    if (int(blockIdx.x) < 5 * u.depth)
        return muon_matrix(u, blockIdx.x, clips, waves);
    // quads: the embedding's 1024, four for each scale, the head's 1024 (the only ones that decay)
    const int quad = (blockIdx.x - 5 * u.depth) * blockDim.x + threadIdx.x, norm = (quad - V * W / 4) >> 2, norms = 2 * u.depth + 1;
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
    const int groups = blockDim.x >> 8, group = threadIdx.x >> 8;
    f32x4 g[UPDATE_GROUPS], part = ZERO;
    const auto request = [&](int first) {
        if (u.norm_parts != 1 && first < u.count)
            part = fold_parts(u, min(first + group, u.count - 1));
#pragma unroll
        for (int n = 0; n < UPDATE_GROUPS; ++n)
            if (n < groups && first + n < u.count)
                g[n] = *reinterpret_cast<const f32x4 *>(u.step[first + n].gradient + at);
    };
    request(0);
    f32x4 m = *reinterpret_cast<const f32x4 *>(u.momentum + at), v = *reinterpret_cast<const f32x4 *>(u.variance + at), w;
#pragma unroll
    for (int k = 0; k < 4; ++k)
        w[k] = master(u.step[0].from.hi, u.step[0].from.lo, at + k);
    for (int first = 0; first < u.count; first += groups) {
        const int steps = min(groups, u.count - first);
        clip_factors(u, first, steps, part, clips, waves);
#pragma unroll
        for (int n = 0; n < UPDATE_GROUPS; ++n) {
            if (n >= steps)
                break;
            const W16Step &step = u.step[first + n];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                float mk = m[k], vk = v[k];
                w[k] = adamw_element(step.adam, decays ? step.adam.weight_decay : 0.f, clips[n], w[k], mk, vk, g[n][k]);
                m[k] = mk, v[k] = vk;
            }
            const auto half = [&](int k, int shift) { return (__float_as_uint(w[k]) >> shift) & 0xffffu; };
            if (live) {
                *reinterpret_cast<u32x2 *>(step.to.hi + at) = u32x2{half(0, 16) | half(1, 16) << 16, half(2, 16) | half(3, 16) << 16};
                *reinterpret_cast<u32x2 *>(step.to.lo + at) = u32x2{half(0, 0) | half(1, 0) << 16, half(2, 0) | half(3, 0) << 16};
            }
        }
        request(first + groups);
        __syncthreads(); // the next clip factors go where these are read
    }
    if (!live)
        return;
    *reinterpret_cast<f32x4 *>(u.momentum + at) = m;
    *reinterpret_cast<f32x4 *>(u.variance + at) = v;
}
int adam_blocks(int depth, int threads) { return (2 * V * W / 4 + 4 * (2 * depth + 1) + threads - 1) / threads; }

void check_shape(int depth, int batch, int context) {
    require(depth >= 1 && depth <= MAX_DEPTH, "w16: depth must be 1..8");
    require(context >= 1 && context <= 8, "w16: context must be 1..8 (the RoPE table has eight entries)");
    require(batch >= 1, "w16: empty batch");
    require(int64_t(batch) * context <= (1 << 24), "w16: too many tokens");
}
Model make_model(int depth, int batch, int context, const uint16_t *hi, const uint16_t *lo) {
    return Model{hi, lo, depth, batch * context, context, tokens_per_wave(context), 0};
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
template <class Kernel> void allow_lds(Kernel kernel, std::atomic<bool> (&configured)[64], size_t bytes = LDS_BYTES) {
    int device = 0;
    check_hip(hipGetDevice(&device));
    require(device >= 0 && device < 64, "w16: device index out of range");
    if (configured[device].load(std::memory_order_acquire))
        return;
    check_hip(hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, int(bytes)),
              "w16 LDS size: ");
    configured[device].store(true, std::memory_order_release);
}
int compute_units() {
    static std::atomic<int> cached[64];
    int device = 0;
    check_hip(hipGetDevice(&device));
    require(device >= 0 && device < 64, "w16: device index out of range");
    int units = cached[device].load(std::memory_order_relaxed);
    if (!units) {
        check_hip(hipDeviceGetAttribute(&units, hipDeviceAttributeMultiprocessorCount, device));
        cached[device].store(units > 0 ? units : 256, std::memory_order_relaxed);
    }
    return units;
}
void launch_weight_gradients(hipStream_t stream, const Model &m, const Workspace &r, const Group &group, int count, bool losses) {
    const int parameters = make_layout(m.depth).count, blocks = fold_blocks(parameters);
    static std::atomic<bool> configured[64];
    allow_lds(w16_weight_gradient_kernel, configured, GRADIENT_LDS);
    hipLaunchKernelGGL(w16_weight_gradient_kernel, dim3((m.depth + 2) * ((r.chunks + 7) / 8 * 8), count), dim3(64 * WAVES), GRADIENT_LDS,
                       stream, m, r, group, parameters);
    hipLaunchKernelGGL(w16_fold_kernel, dim3(blocks + (losses ? m.context : 0), count), dim3(256), 0, stream, r, group, parameters, blocks,
                       m.tokens / m.context, m.context);
    check_hip(hipGetLastError(), "w16 weight gradient launch: ");
}
} // namespace

extern "C" int tgk_w16_forward(hipStream_t stream, int depth, int batch, int context, const uint16_t *weight_hi,
                               const uint16_t *weight_lo, const uint8_t *x, const uint8_t *y, void *workspace,
                               float *token_losses, float *logits, int with_gradient) {
    return guarded([&] {
        check_shape(depth, batch, context);
        require(weight_hi && weight_lo && x && y && workspace && token_losses, "w16_forward: missing operand");
        require(!(reinterpret_cast<uintptr_t>(workspace) & 255), "w16_forward: workspace must be 256-byte aligned");
        Model m = make_model(depth, batch, context, weight_hi, weight_lo);
        const Workspace r = carve(depth, batch, context, workspace);
        const Teams t = pass_teams(r.waves, depth, with_gradient != 0, compute_units());
        m.teams = t.teams;
        static std::atomic<bool> configured[4][64];
        const bool lone = t.roles == 1;
        const auto kernel = with_gradient ? (lone ? w16_forward_kernel<true, 1> : w16_forward_kernel<true, ROLES>)
                                          : (lone ? w16_forward_kernel<false, 1> : w16_forward_kernel<false, ROLES>);
        allow_lds(kernel, configured[(with_gradient != 0) * 2 + lone]);
        hipLaunchKernelGGL(kernel, dim3(t.blocks), dim3(64 * block_waves(t.roles)), t.lds, stream, m, x, y, r, token_losses, logits);
        check_hip(hipGetLastError(), "w16_forward launch: ");
    });
}

extern "C" int tgk_w16_backward(hipStream_t stream, int depth, int batch, int context, const uint16_t *weight_hi,
                                const uint16_t *weight_lo, const uint8_t *x, void *workspace, float *gradient) {
    return guarded([&] {
        check_shape(depth, batch, context);
        require(weight_hi && weight_lo && x && workspace && gradient, "w16_backward: missing operand");
        require(!(reinterpret_cast<uintptr_t>(workspace) & 255), "w16_backward: workspace must be 256-byte aligned");
        Model m = make_model(depth, batch, context, weight_hi, weight_lo);
        const Workspace r = carve(depth, batch, context, workspace);
        const Teams t = pass_teams(r.waves, depth, true, compute_units());
        m.teams = t.teams;
        static std::atomic<bool> configured[2][64];
        const bool lone = t.roles == 1;
        const auto kernel = lone ? w16_backward_kernel<1> : w16_backward_kernel<ROLES>;
        allow_lds(kernel, configured[lone]);
        hipLaunchKernelGGL(kernel, dim3(t.blocks), dim3(64 * block_waves(t.roles)), t.lds, stream, m, r);
        check_hip(hipGetLastError(), "w16_backward launch: ");
        Group group{};
        group.member[0].tokens = const_cast<uint8_t *>(x), group.member[0].workspace = workspace, group.member[0].gradient = gradient;
        launch_weight_gradients(stream, m, r, group, 1, false);
    });
}

int w16_blocks(int batch, int context) {
    return blocks_of(batch, context);
}
int w16_norm_count(int depth) {
    return fold_blocks(make_layout(depth).count) / FOLD_QUARTERS;
}
int w16_norm_parts() {
    return FOLD_QUARTERS;
}
void w16_gradients(hipStream_t stream, int depth, int batch, int context, const W16Data &data, int count, int flying, const W16Batch *batches) {
    require(context == 4 || context == 8, "w16: a training step has a context of 4 or 8");
    require(count >= 1 && count <= W16_BATCHES, "w16: too many batches for one launch");
    Model m = make_model(depth, batch, context, nullptr, nullptr);
    const Workspace r = carve(depth, batch, context, batches[0].workspace);
    Group group{};
    std::copy(batches, batches + count, group.member);
    const Teams t = step_teams(r.waves, count, depth, flying, compute_units());
    m.teams = t.teams;
    static std::atomic<bool> configured[6][64];
    const auto kernel = context == 4 ? (t.roles == 1 ? w16_step_kernel<4, 1, false> : t.rows ? w16_step_kernel<4, ROLES, true> : w16_step_kernel<4, ROLES, false>)
                                     : (t.roles == 1 ? w16_step_kernel<8, 1, false> : t.rows ? w16_step_kernel<8, ROLES, true> : w16_step_kernel<8, ROLES, false>);
    allow_lds(kernel, configured[(context == 8) * 3 + (t.roles == 1 ? 2 : t.rows)]);
    const uint64_t places = uint64_t(data.size) - 8, inverse = places > 1 ? uint64_t((static_cast<unsigned __int128>(1) << 64) / places) : ~uint64_t(0);
    hipLaunchKernelGGL(kernel, dim3(t.blocks, count), dim3(64 * block_waves(t.roles)), t.lds, stream, m, data, inverse, r, group);
    check_hip(hipGetLastError(), "w16_step launch: ");
    launch_weight_gradients(stream, m, r, group, count, true);
}
void w16_updates(hipStream_t stream, int depth, float *momentum, float *variance, int norm_count, int norm_parts, int count,
                 const W16Step *steps) {
    require(norm_parts == 1 ? count == 1 : norm_count <= 64, "w16: a fold's norms have a lane each");
    for (int i = 1; i < count; ++i)
        require(steps[i].muon.ns_steps == steps[0].muon.ns_steps && (steps[i].adam.clip > 0.f) == (steps[0].adam.clip > 0.f), "w16: steps of one launch are alike");
    require(count >= 1 && count <= W16_BATCHES, "w16: too many steps for one launch");
    Update u{momentum, variance, norm_count, norm_parts, depth, count, steps[0].muon.ns_steps, {}};
    std::copy(steps, steps + count, u.step);
    const int threads = 256 * std::min(count, UPDATE_GROUPS);
    hipLaunchKernelGGL(w16_update_kernel, dim3(5 * depth + adam_blocks(depth, threads)), dim3(threads), 0, stream, u);
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
        Update u{momentum, nullptr, norm_count, 1, depth, 1, ns_steps, {}};
        u.step[0] = {weights, weights, gradient, norm_partials, adam, MuonArgs{lr, momentum_rate, weight_decay, ns_steps}};
        hipLaunchKernelGGL(w16_update_kernel, dim3(5 * depth), dim3(256), 0, stream, u); // the matrices' blocks alone
        check_hip(hipGetLastError(), "w16_muon launch: ");
    });
}
