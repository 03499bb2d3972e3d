// Engine behind the tg_* C ABI: owns every device buffer, and runs the training step as a
// sequence of kernel launches on one HIP stream.  Host-side counterpart of the reference's
// cuda/runtime.cu + cuda/engine_state.cu (resource ownership, transfers, entry points) and of the
// op sequencing that its persistent kernel does on the device (cuda/trainer.cuh:103-125,
// cuda/model.cuh:8-99).  All arithmetic is in the tgk_* kernels; this file only sequences them.
#include "common.h"
#include "gemm_list.h"
#include "readback.h"
#include "step.h"
#include "width16.h"
#include "width16_launch.h"
#include "../../include/tg_model.h"
#include "../../include/tgk_kernels.h"
#include <algorithm>
#include <climits>
#include <cmath>
#include <cstring>
#include <vector>

namespace {

constexpr int MaxLaunchSteps = 4096; // cuda/types.cuh:10
constexpr int NormPartials = 1024;
constexpr int ListUnit = 128;   // every width is a multiple of it (wgrad_list)
constexpr int RowTile = 128;    // smallest number of rows the matrix products take
constexpr int HardwareQueues = 4; // of the process, the runtime's default: as many streams run side by side
constexpr int MaxInFlight = 16; // batches in flight, each with its own stream and saved activations
// Rows of the loss history, a ring over the steps: two steps that share a row are at least MaxInFlight apart, so the later
// one is behind the earlier one also where they are in different launches and on different streams.
constexpr int HistoryRows = MaxLaunchSteps + MaxInFlight;

struct LayerBuffers {
    bf16_t *n1, *qkv, *o, *mid, *n2, *u, *a;
    float *lse;
};

void ok(int status) {
    if (status < 0)
        throw std::runtime_error(tg_last_error);
}
// one operator launch, attributed to a TG_CLASS_* for tg_profile_step
#define OP(cls, call)                 \
    do {                              \
        Scope profile_scope(this, cls); \
        ok(call);                     \
    } while (0)

// optim.h:18-44
StepRates onecycle_point(const OneCycle &s, int step) {
    if (s.total_steps < 1 || step < 0 || step >= s.total_steps ||
        !(s.warmup_fraction > 0 && s.warmup_fraction < 1) ||
        !(s.initial_lr_fraction > 0 && s.initial_lr_fraction < 1) ||
        !(s.final_lr_fraction > 0 && s.final_lr_fraction <= s.initial_lr_fraction) ||
        !(s.low_momentum >= 0 && s.low_momentum < 1) ||
        !(s.high_momentum >= s.low_momentum && s.high_momentum < 1))
        throw std::runtime_error("Invalid OneCycle schedule or step");
    const double warmup_steps = s.warmup_fraction * s.total_steps - 1;
    if (warmup_steps == 0)
        throw std::runtime_error("OneCycle warmup must span at least two steps");
    const bool warming = step <= warmup_steps;
    const double fraction =
        warming ? step / warmup_steps : (step - warmup_steps) / (s.total_steps - 1 - warmup_steps);
    const double c = 0.5 * (1 + std::cos(3.14159265358979323846 * fraction));
    const auto between = [c](double from, double to) { return to + (from - to) * c; };
    return {float(warming ? between(s.initial_lr_fraction, 1.0) : between(1.0, s.final_lr_fraction)),
            float(warming ? between(s.high_momentum, s.low_momentum)
                          : between(s.low_momentum, s.high_momentum))};
}

} // namespace

// Everything one batch in flight owns: its stream, its tokens, its saved activations and its gradient.
// Slot 0 is on the engine's stream (a synchronous engine has no other); inflight = K gives K slots on K streams
// (the worker teams of cuda/pipeline.cuh:52-92).
struct Slot {
    hipStream_t stream = nullptr;
    uint8_t *input = nullptr, *target = nullptr;
    float *token_losses = nullptr, *gradient = nullptr;
    std::vector<bf16_t *> x; // x[l] = input of block l; x[depth] = output of the last block
    std::vector<LayerBuffers> layers;
    bf16_t *nf = nullptr, *logits = nullptr, *t1 = nullptr;
    // All weight gradients of a step go out as one launch behind the backward pass: every block keeps the four
    // output gradients that launch reads: g_x[l] = gradient of the loss by x[l] (g_x[l + 1] enters block l), g_mid[l]
    // by the block's middle, g_u[l] by the MLP pre-activation, g_qkv[l] by the packed projections.  Where the device
    // has no room for that, all blocks share one set of the four (g_x: one buffer) and every block's weight gradients
    // are a launch of their own, behind its attention.
    std::vector<bf16_t *> g_x, g_mid, g_u, g_qkv;
    std::vector<TgkWgradJob> wgrad_jobs; // four a block, the head, the token table
    struct WgradLaunch {
        int first, count; // of wgrad_jobs
        void *table;
    };
    std::vector<WgradLaunch> wgrads; // one; or one a block, the head's and the token table's
    bf16_t *onehot = nullptr; // [tokens][256]: the token table's gradient is one more product of that launch
    // ... and the kernels that write the gradient leave the sums of its squares here (cuda/trainer.cuh:35-46): the
    // launch above for the matrices and, of the gradients that are there already, for the ranges in `norm_ranges` (every other
    // tensor), which are a launch of their own where the tiles are large
    float *norms = nullptr;
    int list_norms = 0, range_norms = 0;
    void *norm_ranges = nullptr;
    void *workspace = nullptr;
    // LayerNorm parameter gradients: every LayerNorm backward of a step leaves its per-block partial sums in a
    // block of its own here and one launch at the end of the backward pass folds all 2 * depth + 1 of them
    uint8_t *ln_partials = nullptr;
    void *ln_targets = nullptr; // device array of {dgamma, dbeta} pointers into `gradient`, in fold order
};
// One immutable copy of the weights: a batch reads a single version from its first kernel to its last
// (cuda/pipeline.cuh:36-38).  inflight = K keeps K + 1 of them in a ring; a synchronous engine one.
struct Version {
    uint16_t *hi = nullptr, *lo = nullptr;
    uint16_t *t = nullptr;     // every matrix of hi transposed ([In][Out]), same offsets (wide model only)
    hipEvent_t done = nullptr; // the optimizer step that wrote this version has finished
};

struct Engine {
    TgModelConfig config{};
    TgParameterLayout layout{};
    hipStream_t stream = nullptr;
    hipStream_t second = nullptr; // of large results
    hipEvent_t branched = nullptr;
    std::vector<void *> allocations;
    size_t allocated_bytes = 0;
    int compute_units = 0;
    bool width16 = false; // the reference's own network, created from the plain Config

    std::vector<Slot> slots;
    std::vector<Version> versions;
    void *transpose_jobs = nullptr;
    int transpose_count = 0, transpose_tiles = 0;
    float *momentum = nullptr, *variance = nullptr;
    float *norm_partials = nullptr, *loss_history = nullptr;
    int64_t *segment_starts = nullptr;
    uint8_t *segment_flags = nullptr;
    int segments = 0;
    uint8_t *data = nullptr;
    int64_t data_size = 0;
    float *logits_f32 = nullptr;
    size_t workspace_bytes = 0;

    std::shared_ptr<Readback> readback; // of the engine's device
    float *batch_means = nullptr; // [context]: the per-position losses of a fixed batch

    std::vector<StepRates> schedule;
    uint64_t step = 0;
    uint64_t floor = 0; // oldest weight version that exists: the step at the last tg_set_weights / _set_optimizer_state
    // the version that the last shared launch left (train_width16), or `floor`: the steps up to it are on the engine's stream
    uint64_t shared_end = 0;
    bool shared_recorded = false; // whether that version's event has been recorded behind it
    int last_train_steps = 0;
    uint64_t last_train_first = 0;
    std::vector<int> version_trace; // weight version each step of the last tg_train read
    uint64_t total_staleness = 0;
    int max_staleness = 0;

    // optional per-class timing of one step (tg_profile_step): event pairs around every launch
    struct Span {
        int cls;
        hipEvent_t start, stop;
    };
    bool profiling = false;
    std::vector<Span> spans;
    std::vector<hipEvent_t> event_pool;
    hipEvent_t event() {
        if (event_pool.empty()) {
            hipEvent_t fresh;
            check_hip(hipEventCreate(&fresh));
            return fresh;
        }
        hipEvent_t pooled = event_pool.back();
        event_pool.pop_back();
        return pooled;
    }
    struct Scope {
        Engine *e;
        size_t index = 0;
        Scope(Engine *engine, int cls) : e(engine) { // profiling exists for synchronous engines: one stream
            if (!e->profiling)
                return;
            index = e->spans.size();
            e->spans.push_back({cls, e->event(), e->event()});
            check_hip(hipEventRecord(e->spans[index].start, e->stream));
        }
        ~Scope() {
            if (e->profiling)
                (void)hipEventRecord(e->spans[index].stop, e->stream);
        }
    };

    float *history_row(uint64_t at) const { return loss_history + size_t(at % HistoryRows) * config.base.context; }
    int tokens() const { return config.base.batch * config.base.context; }

    template <class T> void allocate(T *&ptr, size_t n, bool zero = true) { // cuda/engine_internal.h:17-27
        void *raw = nullptr;
        check_hip(hipMalloc(&raw, n * sizeof(T)), "allocation: ");
        ptr = static_cast<T *>(raw);
        allocations.push_back(raw);
        allocated_bytes += n * sizeof(T);
        if (zero)
            check_hip(hipMemsetAsync(raw, 0, n * sizeof(T), stream));
    }
    // gives back every allocation behind the first `count`
    void release_after(size_t count, size_t bytes) {
        (void)hipStreamSynchronize(stream);
        for (; allocations.size() > count; allocations.pop_back())
            (void)hipFree(allocations.back());
        allocated_bytes = bytes;
    }
    void use_device() const { check_hip(hipSetDevice(config.base.device)); }
    void sync_slots() const { // every slot's stream but the engine's own
        for (const Slot &slot : slots)
            if (slot.stream && slot.stream != stream)
                check_hip(hipStreamSynchronize(slot.stream));
    }
    void sync() const { // every stream: the engine is quiescent afterwards
        sync_slots();
        check_hip(hipStreamSynchronize(stream));
    }
    Version &current() { return versions[step % versions.size()]; }
    template <class T> void upload(T *device, const T *host, size_t n) {
        check_hip(hipMemcpyAsync(device, host, n * sizeof(T), hipMemcpyHostToDevice, stream));
    }
    // results to the caller's memory, behind everything on the engine's stream; returns when they are there
    void download(const std::vector<ReadbackPiece> &pieces) {
        size_t bytes = 0;
        for (const ReadbackPiece &piece : pieces)
            bytes += piece.bytes;
        const bool large = bytes >= Readback::LARGE;
        if (large) {
            if (!second)
                check_hip(hipStreamCreate(&second)); // default priority
            if (!branched)
                check_hip(hipEventCreateWithFlags(&branched, hipEventDisableTiming));
            check_hip(hipEventRecord(branched, stream));
            check_hip(hipStreamWaitEvent(second, branched, 0));
        }
        readback->fetch(stream, pieces, large ? second : nullptr);
    }
    ~Engine() { // cuda/engine_internal.h:28-37
        (void)hipSetDevice(config.base.device);
        for (Slot &slot : slots)
            if (slot.stream && slot.stream != stream)
                (void)hipStreamSynchronize(slot.stream);
        if (stream)
            (void)hipStreamSynchronize(stream);
        if (second)
            (void)hipStreamSynchronize(second);
        for (void *allocation : allocations)
            (void)hipFree(allocation);
        for (Slot &slot : slots) {
            if (slot.stream && slot.stream != stream)
                (void)hipStreamDestroy(slot.stream);
        }
        for (Version &version : versions)
            if (version.done)
                (void)hipEventDestroy(version.done);
        for (Span &span : spans) {
            (void)hipEventDestroy(span.start);
            (void)hipEventDestroy(span.stop);
        }
        for (hipEvent_t pooled : event_pool)
            (void)hipEventDestroy(pooled);
        if (branched)
            (void)hipEventDestroy(branched);
        if (second)
            (void)hipStreamDestroy(second);
        if (stream)
            (void)hipStreamDestroy(stream);
    }

    // input gradients and the head's forward projection read the transposed weights: call after every change of a
    // version's hi half
    void refresh_transposed(const Version &v) {
        if (width16)
            return;
        ok(tgk_transpose_batch(stream, v.hi, v.t, transpose_jobs, transpose_count, transpose_tiles));
    }

    // cuda/model.cuh:8-59.  evaluate: logits stay logits; otherwise they are replaced by dlogits.
    // On the slot's stream, with one weight version, from the slot's first `batch` sequences.  last_position: one
    // sequence, and only the logits of its last position are wanted (`logits_out` receives that row): behind the
    // attention of the last block nothing but the last tile of rows is computed.
    // embedded: the slot's tokens have already been drawn and embedded (sample_embed).
    void forward(Slot &s, const Version &v, bool with_gradient, float *logits_out, int batch, bool last_position = false,
                 bool embedded = false) {
        const Config &c = config.base;
        hipStream_t stream = s.stream;
        const uint8_t *tokens_in = s.input, *targets = s.target;
        float *token_losses = s.token_losses;
        if (width16) {
            OP(TG_CLASS_OTHER, tgk_w16_forward(stream, c.depth, batch, c.context, v.hi, v.lo, tokens_in, targets,
                                               s.workspace, token_losses, logits_out, with_gradient ? 1 : 0));
            return;
        }
        const auto w = [&](int64_t offset) { return v.hi + offset; };
        const auto wl = [&](int64_t offset) { return v.lo + offset; };
        const auto wt = [&](int64_t offset) { return v.t + offset; };
        std::vector<bf16_t *> &x = s.x;
        std::vector<LayerBuffers> &layers = s.layers;
        bf16_t *nf = s.nf, *logits = s.logits;
        const int d = config.d_model, F = config.ffn, V = config.vocab, T = c.context;
        const float scale = 1.0f / std::sqrt(float(d / config.heads));
        int M = batch * T;
        if (!embedded)
            OP(TG_CLASS_OTHER, tgk_embed_fwd(stream, M, T, d, tokens_in, w(layout.embedding), w(layout.positions), x[0]));
        for (int l = 0; l < c.depth; ++l) {
            const TgLayerParameters &p = layout.layers[l];
            // without a backward pass every layer writes where the first one did: the Infinity Cache then holds the weights from one
            // pass to the next
            const LayerBuffers &b = layers[with_gradient ? l : 0];
            const bf16_t *from = x[with_gradient ? l : l & 1];
            bf16_t *to = x[with_gradient ? l + 1 : (l + 1) & 1];
            OP(TG_CLASS_LAYERNORM_FWD, tgk_layernorm_fwd(stream, M, d, from, w(p.ln1_g), wl(p.ln1_g), w(p.ln1_b), wl(p.ln1_b), b.n1,
                                 config.ln_eps));
            OP(TG_CLASS_GEMM_FWD, tgk_gemm_fwd(stream, M, 3 * d, d, b.n1, d, w(p.qkv), d, b.qkv, 3 * d, nullptr, 0, nullptr, 0));
            OP(TG_CLASS_ATTN_FWD, tgk_attn_fwd(stream, batch, config.heads, T, d / config.heads, b.qkv, b.qkv + d, b.qkv + 2 * d,
                            3 * d, b.o, d, b.lse, scale));
            const size_t skip = last_position && l == c.depth - 1 ? size_t(M - RowTile) : 0; // rows nobody reads
            M -= int(skip);
            const bf16_t *o = b.o + skip * d, *in = from + skip * d;
            OP(TG_CLASS_GEMM_FWD, tgk_gemm_fwd(stream, M, d, d, o, d, w(p.attn_out), d, b.mid, d, in, d, nullptr, 0));
            OP(TG_CLASS_LAYERNORM_FWD, tgk_layernorm_fwd(stream, M, d, b.mid, w(p.ln2_g), wl(p.ln2_g), w(p.ln2_b), wl(p.ln2_b), b.n2,
                                 config.ln_eps));
            if (with_gradient)
                OP(TG_CLASS_GEMM_FWD_GELU, tgk_gemm_fwd(stream, M, F, d, b.n2, d, w(p.mlp_up), d, b.u, F, nullptr, 0, b.a, F));
            else
                OP(TG_CLASS_GEMM_FWD_GELU, gemm_fwd_gelu_only(stream, M, F, d, b.n2, d, w(p.mlp_up), d, b.a, F));
            OP(TG_CLASS_GEMM_FWD, tgk_gemm_fwd(stream, M, d, F, b.a, F, w(p.mlp_down), F, to, d, b.mid, d, nullptr, 0));
        }
        OP(TG_CLASS_LAYERNORM_FWD, tgk_layernorm_fwd(stream, M, d, x[with_gradient ? c.depth : c.depth & 1], w(layout.lnf_g), wl(layout.lnf_g), w(layout.lnf_b),
                             wl(layout.lnf_b), nf, config.ln_eps));
        OP(TG_CLASS_HEAD, tgk_gemm_fwd_t(stream, M, V, d, nf, d, wt(layout.head), V, logits, V, nullptr, 0, nullptr, 0));
        const size_t row = last_position ? size_t(M - 1) : 0; // the first row whose logits are wanted
        OP(TG_CLASS_OTHER, tgk_cross_entropy(stream, M - int(row), V, logits + row * V, targets, token_losses, logits_out,
                             1.0f / float(M), with_gradient ? 1 : 0));
    }

    // cuda/model.cuh:61-99.  Every element of `gradient` is overwritten: nothing needs zeroing.  means: where the batch's
    // losses per position go.
    void backward(Slot &s, const Version &v, float *means) {
        const Config &c = config.base;
        hipStream_t stream = s.stream;
        const uint8_t *tokens_in = s.input;
        float *gradient = s.gradient;
        void *workspace = s.workspace;
        if (width16) {
            OP(TG_CLASS_OTHER, tgk_w16_backward(stream, c.depth, c.batch, c.context, v.hi, v.lo, tokens_in, workspace,
                                                gradient));
            OP(TG_CLASS_OTHER, tgk_position_means(stream, s.token_losses, c.batch, c.context, means));
            return;
        }
        const auto w = [&](int64_t offset) { return v.hi + offset; };
        const auto wl = [&](int64_t offset) { return v.lo + offset; };
        const auto wt = [&](int64_t offset) { return v.t + offset; };
        std::vector<bf16_t *> &x = s.x;
        std::vector<LayerBuffers> &layers = s.layers;
        bf16_t *logits = s.logits, *t1 = s.t1;
        const int M = tokens(), d = config.d_model, F = config.ffn, V = config.vocab, T = c.context;
        const float scale = 1.0f / std::sqrt(float(d / config.heads));
        float *g = gradient;
        // LayerNorm j of the fold: 0 = final, 1 + 2 l = block l's second, 2 + 2 l = its first
        const size_t ln_stride = tgk_layernorm_bwd_workspace(M, d);
        const auto ln_rows = [&](int job, const bf16_t *input, const bf16_t *dy, int64_t gamma, const bf16_t *residual,
                                 bf16_t *dx) {
            return tgk_layernorm_bwd_rows(stream, M, d, input, dy, w(gamma), wl(gamma), residual, dx, config.ln_eps,
                                          s.ln_partials + size_t(job) * ln_stride, ln_stride);
        };
        // No weight gradient in the loop: every block leaves its output gradients in buffers of its own and one
        // launch at the end computes all 4 * depth + 2 products (the head's included - its operands are dlogits,
        // still in `logits`, and nf - and the token table's, one-hot^T times the gradient entering the first block).
        // Or, where those buffers did not fit, a launch behind the head's input gradient, one in every block, before
        // the block's last kernel overwrites the gradient that entered it, and one at the end.
        const bool together = s.wgrads.size() == 1, norms = together && c.clip > 0;
        const SumsqSegments ranges = norms ? SumsqSegments{g, static_cast<const SumsqSegment *>(s.norm_ranges), s.range_norms,
                                                           s.norms + s.list_norms}
                                           : SumsqSegments{};
        const auto weight_gradients = [&](const Slot::WgradLaunch &part) {
            Scope profile_scope(this, TG_CLASS_GEMM_WGRAD);
            return wgrad_list(stream, M, part.count, s.wgrad_jobs.data() + part.first, ListUnit, part.table, workspace,
                              workspace_bytes, norms ? s.norms : nullptr, ranges);
        };
        OP(TG_CLASS_HEAD, tgk_gemm_dgrad_t(stream, M, V, d, logits, V, wt(layout.head), V, t1, d, nullptr, 0));
        if (!together)
            weight_gradients(s.wgrads[c.depth]);
        OP(TG_CLASS_LAYERNORM_BWD, ln_rows(0, x[c.depth], t1, layout.lnf_g, nullptr, s.g_x[c.depth]));
        for (int l = c.depth - 1; l >= 0; --l) {
            const TgLayerParameters &p = layout.layers[l];
            LayerBuffers &b = layers[l];
            bf16_t *in = s.g_x[l + 1], *mid = s.g_mid[l], *gu = s.g_u[l], *gqkv = s.g_qkv[l];
            OP(TG_CLASS_GEMM_DGRAD_GELU, tgk_gemm_dgrad_t(stream, M, d, F, in, d, wt(p.mlp_down), d, gu, F, b.u, F));
            OP(TG_CLASS_GEMM_DGRAD, tgk_gemm_dgrad_t(stream, M, F, d, gu, F, wt(p.mlp_up), F, t1, d, nullptr, 0));
            OP(TG_CLASS_LAYERNORM_BWD, ln_rows(1 + 2 * l, b.mid, t1, p.ln2_g, in, mid));
            OP(TG_CLASS_GEMM_DGRAD, tgk_gemm_dgrad_t(stream, M, d, d, mid, d, wt(p.attn_out), d, t1, d, nullptr, 0));
            OP(TG_CLASS_ATTN_BWD, tgk_attn_bwd(stream, c.batch, config.heads, T, d / config.heads, b.qkv, b.qkv + d,
                                               b.qkv + 2 * d, 3 * d, b.o, d, b.lse, t1, d, gqkv, gqkv + d, gqkv + 2 * d,
                                               3 * d, scale, workspace, workspace_bytes));
            if (!together)
                weight_gradients(s.wgrads[l]);
            OP(TG_CLASS_GEMM_DGRAD, tgk_gemm_dgrad_t(stream, M, 3 * d, d, gqkv, 3 * d, wt(p.qkv), 3 * d, t1, d, nullptr, 0));
            OP(TG_CLASS_LAYERNORM_BWD, ln_rows(2 + 2 * l, x[l], t1, p.ln1_g, mid, s.g_x[l]));
        }
        OP(TG_CLASS_OTHER, backward_rest(stream, {c.batch, T, d, tokens_in, s.g_x[0], s.onehot, g + layout.positions,
                                                  reinterpret_cast<const float *>(s.ln_partials), ln_stride / sizeof(float),
                                                  2 * c.depth + 1, 0, s.ln_targets, s.token_losses, means}));
        const bool summed = weight_gradients(s.wgrads.back());
        if (norms && !summed)
            OP(TG_CLASS_OPTIMIZER, tgk_sumsq_segments(stream, g, ranges.segments, ranges.count, ranges.partials));
    }

    // learning rates and momenta of optimizer step `at` (0-based)
    struct Rates {
        float lr, beta1, muon_lr, muon_momentum;
    };
    Rates rates(uint64_t at) const {
        const Config &c = config.base;
        if (schedule.empty())
            return {c.learning_rate, c.beta1, c.muon_lr, c.momentum};
        // cuda/optim.cuh:81-88: one point drives both learning rates and both momenta
        const StepRates &point = schedule[at];
        return {c.learning_rate * point.multiplier, point.momentum, c.muon_lr * point.multiplier, point.momentum};
    }
    W16Step w16_step(uint64_t at, const float *gradient, const float *norms, const Version &now, const Version &to) const {
        const Config &c = config.base;
        const Rates r = rates(at);
        return {{now.hi, now.lo}, {to.hi, to.lo}, gradient, norms,
                adam_args(r.lr, r.beta1, c.beta2, c.epsilon, c.weight_decay, c.clip, at),
                {r.muon_lr, r.muon_momentum, c.weight_decay, c.ns_steps}};
    }

    // cuda/optim.cuh:66-106 for optimizer step `at` (0-based), on `stream`: gradient -> the weights of version `to`, from
    // the previous version's, `now`.
    // `from`: the slot whose backward pass has just written `gradient`, when it left the sums of squares with it
    void optimize(hipStream_t stream, uint64_t at, const float *gradient, const Version &now, Version &to,
                  const Slot *from = nullptr) {
        const Config &c = config.base;
        uint16_t *weight_hi = to.hi, *weight_lo = to.lo, *weight_t = to.t;
        const bool fused = from && from->norms;
        if (c.clip > 0 && !fused)
            OP(TG_CLASS_OPTIMIZER, tgk_sumsq_partials(stream, gradient, size_t(layout.count), norm_partials, NormPartials));
        const float *norms = fused ? from->norms : norm_partials;
        const int norm_count = fused ? from->list_norms + from->range_norms : NormPartials;
        if (width16) { // AdamW's tensors and the hidden matrices (cuda/optim.cuh:92-118)
            const W16Step step = w16_step(at, gradient, norms, now, to);
            w16_updates(stream, c.depth, momentum, variance, norm_count, 1, 1, &step);
            return;
        }
        const Rates r = rates(at);
        if (&now != &to) {
            const size_t bytes = size_t(layout.count) * 2;
            check_hip(hipMemcpyAsync(to.hi, now.hi, bytes, hipMemcpyDeviceToDevice, stream));
            check_hip(hipMemcpyAsync(to.lo, now.lo, bytes, hipMemcpyDeviceToDevice, stream));
        }
        OP(TG_CLASS_OPTIMIZER, tgk_adamw(stream, size_t(layout.count), weight_hi, weight_lo, momentum, variance, gradient,
                     norms, norm_count, segment_starts, segment_flags, segments, r.lr, r.beta1, c.beta2, c.epsilon, c.weight_decay,
                     c.clip, at));
        OP(TG_CLASS_OPTIMIZER, tgk_transpose_batch(stream, weight_hi, weight_t, transpose_jobs, transpose_count,
                                                   transpose_tiles));
    }
    // batch `at`: sample, forward, loss row, backward, on one slot with one weight version
    void batch_gradient(Slot &s, const Version &v, uint64_t at) {
        const Config &c = config.base;
        hipStream_t stream = s.stream;
        OP(TG_CLASS_OTHER, sample_embed(stream, data, data_size, c.seed, at, c.batch, c.context, config.d_model, s.input, s.target,
                                        v.hi + layout.embedding, v.hi + layout.positions, s.x[0]));
        forward(s, v, true, nullptr, c.batch, false, true);
        backward(s, v, history_row(at));
    }
    // Whether the batches of a call of `steps` steps share their launches.
    bool shares_launches(int steps) const {
        const Config &c = config.base;
        return w16::shares_launches(c.depth, int(slots.size()), flying(), w16_blocks(c.batch, c.context), steps, compute_units);
    }
    int flying() const { return std::min(int(slots.size()), HardwareQueues); } // batches on streams of their own that run side by side
    // Training steps of the width-16 network from `at` on; returns how many.  Batch s reads the weights of version
    // max(floor, s - K + 1), whichever way it is launched.
    // `shared`: up to K batches go out as one launch of each kernel on the engine's stream, and their optimizer steps as one
    // more.  The versions that they read are there before the first of those, as batch s reads nothing newer than `at`.
    // Otherwise one batch and its optimizer step, on its slot's stream, as the wide model's below.  Its slot is free, and
    // the version that it reads is there, behind step at - K: that ran on this stream, or shared a launch, whose last one left
    // version shared_end.
    int train_width16(uint64_t at, int most, bool shared, int *trace) {
        const Config &c = config.base;
        const uint64_t K = slots.size(), ring = versions.size();
        const int count = shared ? int(std::min<uint64_t>(K, uint64_t(most))) : 1;
        W16Batch batches[MaxInFlight];
        W16Step steps[MaxInFlight];
        for (int i = 0; i < count; ++i) {
            const uint64_t step = at + uint64_t(i), read = K == 1 ? step : std::max(floor, step + 1 >= K ? step + 1 - K : 0);
            const Slot &s = slots[step % K];
            const Version &v = versions[read % ring];
            batches[i] = {{v.hi, v.lo}, step, s.input, s.workspace, s.token_losses, history_row(step), s.gradient, s.norms};
            steps[i] = w16_step(step, s.gradient, s.norms, versions[step % ring], versions[(step + 1) % ring]);
            trace[i] = int(read);
            total_staleness += step - read;
            max_staleness = std::max(max_staleness, int(step - read));
        }
        const hipStream_t on = shared ? stream : slots[at % K].stream;
        const auto wait_for = [&](uint64_t version) { check_hip(hipStreamWaitEvent(on, versions[version % ring].done, 0)); };
        if (shared && K > 1 && at != shared_end) // the steps before ran on their slots' streams
            wait_for(at);
        if (!shared && at < shared_end + K) {
            if (!shared_recorded) // an event costs every shared launch 2 us, and only the first step off the stream needs one
                check_hip(hipEventRecord(versions[shared_end % ring].done, stream));
            shared_recorded = true;
            wait_for(shared_end);
        }
        {
            Scope profile_scope(this, TG_CLASS_OTHER);
            w16_gradients(on, c.depth, c.batch, c.context, {data, data_size, c.seed}, count, shared ? 1 : flying(), batches);
        }
        if (!shared && at != shared_end)
            wait_for(at);
        {
            Scope profile_scope(this, TG_CLASS_OPTIMIZER);
            w16_updates(on, c.depth, momentum, variance, slots[0].list_norms, w16_norm_parts(), count, steps);
        }
        if (shared)
            shared_end = at + uint64_t(count), shared_recorded = false;
        else
            check_hip(hipEventRecord(versions[(at + 1) % ring].done, on));
        return count;
    }
    // One training step of the wide model.  Synchronous engine: everything in order on the one stream, weights updated in place
    // (cuda/trainer.cuh:109-124).  inflight = K (cuda/pipeline.cuh:40-126 as streams and events): batch `at` and its
    // optimizer step run on the stream of slot at % K, behind optimizer step at - K.  That order alone lets the batch
    // read max(floor, at - K + 1), the oldest version the ring still guarantees, and frees the slot's gradient.  The
    // optimizer step waits for its predecessor, on another slot's stream; the version that it overwrites, at - K, was
    // last read by batch at - 1, which that predecessor follows.  Optimizer steps on a stream of their own (K + 1
    // streams) cost two more events a step and shared one of the process's four hardware queues with a slot at K = 4.  The
    // choice is made on the host, so a run is reproducible; the staleness bound at - K + 1 <= version <= at is the
    // reference's.
    void train_step(uint64_t at, int *trace) {
        const uint64_t K = slots.size(), ring = versions.size();
        if (K == 1) {
            batch_gradient(slots[0], versions[0], at);
            optimize(stream, at, slots[0].gradient, versions[0], versions[0], &slots[0]);
            *trace = int(at);
            return;
        }
        Slot &s = slots[at % K];
        const uint64_t read = std::max(floor, at + 1 >= K ? at + 1 - K : 0);
        batch_gradient(s, versions[read % ring], at);
        const Version &from = versions[at % ring];
        Version &to = versions[(at + 1) % ring];
        check_hip(hipStreamWaitEvent(s.stream, from.done, 0));
        optimize(s.stream, at, s.gradient, from, to, &s);
        check_hip(hipEventRecord(to.done, s.stream));
        *trace = int(read);
        total_staleness += at - read;
        max_staleness = std::max(max_staleness, int(at - read));
    }
    void train(uint64_t at, int steps, int *trace) {
        const bool shared = width16 && shares_launches(steps);
        for (int i = 0; i < steps;) {
            if (width16)
                i += train_width16(at + uint64_t(i), steps - i, shared, trace + i);
            else
                train_step(at + uint64_t(i), trace + i), ++i;
        }
    }
};

namespace {

void validate(const TgModelConfig &m) {
    const Config &c = m.base;
    if (c.depth < 1 || c.depth > TG_MAX_DEPTH)
        throw std::runtime_error("Supported: depth 1..64");
    if (m.vocab != 256)
        throw std::runtime_error("Supported: vocabulary 256 (byte tokens)");
    if (m.d_model < 128 || m.d_model % 128 || m.d_model > 2048)
        throw std::runtime_error("Supported: d_model a multiple of 128, at most 2048");
    if (m.heads * 64 != m.d_model)
        throw std::runtime_error("Supported: head_dim 64 (heads = d_model / 64)");
    if (m.ffn < 128 || m.ffn % 128)
        throw std::runtime_error("Supported: ffn a multiple of 128");
    if (c.context < 128 || c.context % 128)
        throw std::runtime_error("Supported: context a multiple of 128");
    if (c.batch < 1 || int64_t(c.batch) * c.context > (int64_t(1) << 24))
        throw std::runtime_error("Supported: batch >= 1 with batch*context <= 2^24 tokens");
    if (c.inflight < 1 || c.inflight > MaxInFlight)
        throw std::runtime_error("inflight must be 1.." + std::to_string(MaxInFlight));
    if (!(m.ln_eps > 0))
        throw std::runtime_error("ln_eps must be positive");
}

// The engine's stream, which is slot 0's, and one for every further slot.  The runtime has a few hardware queues, makes them as
// streams come and then gives each new stream the one that has the fewest, so streams made one behind another have
// different ones, but only once every queue is there and has as many: two slots that share one run one behind the other.  So as
// many streams are made first, and given back.  Depth 8, 768 sequences of 8, K = 4, calls of one step, us a step without and with them:
// alone 36, 36; beside another engine or two, after one that is gone, with torch at work 49 to 51, 33 to 36.  K = 2 beside two others 80, 48.
// They make the engine's creation longer, K = 2 / 4 / 8 0.2, 0.4, 1.2 -> 1.5, 2.8, 4.2 ms, as much as 100 to 200 steps give back.
void build_streams(Engine *e, int inflight) {
    struct Spare {
        std::vector<hipStream_t> streams;
        ~Spare() {
            for (hipStream_t stream : streams)
                (void)hipStreamDestroy(stream);
        }
    } spare;
    hipStream_t made = nullptr;
    while (inflight > 1 && spare.streams.size() < HardwareQueues && hipStreamCreate(&made) == hipSuccess)
        spare.streams.push_back(made);
    (void)hipGetLastError(); // one that is not to be had is no later call's error
    e->slots.resize(size_t(inflight));
    for (Slot &slot : e->slots) {
        check_hip(hipStreamCreate(&slot.stream)); // default priority
        if (&slot == &e->slots[0])
            e->stream = slot.stream;
    }
}

// Events, staging memory and the buffers every model kind needs per slot and per weight version.
void build_slots(Engine *e, int inflight, bool transposed_copies) {
    const size_t P = size_t(e->layout.count), M = size_t(e->tokens());
    e->readback = Readback::shared(e->config.base.device);
    e->versions.resize(inflight > 1 ? size_t(inflight) + 1 : 1);
    for (Slot &slot : e->slots) {
        e->allocate(slot.input, M);
        e->allocate(slot.target, M);
        e->allocate(slot.token_losses, M);
        e->allocate(slot.gradient, P);
    }
    for (Version &version : e->versions) {
        e->allocate(version.hi, P);
        e->allocate(version.lo, P);
        if (transposed_copies)
            e->allocate(version.t, P);
        if (inflight > 1)
            check_hip(hipEventCreateWithFlags(&version.done, hipEventDisableTiming));
    }
}

void build_transpose_jobs(Engine *e) {
    struct Job {
        int64_t offset;
        int rows, cols, first_tile, pad;
    };
    std::vector<Job> jobs;
    int tiles = 0;
    const auto add = [&](int64_t offset, int rows, int cols) {
        jobs.push_back({offset, rows, cols, tiles, 0});
        tiles += (rows / 64) * (cols / 64);
    };
    const TgParameterLayout &p = e->layout;
    const int d = e->config.d_model, F = e->config.ffn, V = e->config.vocab;
    for (int l = 0; l < e->config.base.depth; ++l) {
        const TgLayerParameters &b = p.layers[l];
        add(b.qkv, 3 * d, d);
        add(b.attn_out, d, d);
        add(b.mlp_up, F, d);
        add(b.mlp_down, d, F);
    }
    add(p.head, V, d);
    Job *device = nullptr;
    e->allocate(device, jobs.size(), false);
    e->upload(device, jobs.data(), jobs.size());
    e->sync();
    e->transpose_jobs = device;
    e->transpose_count = int(jobs.size());
    e->transpose_tiles = tiles;
}

void build_segments(Engine *e) {
    // weight-decay groups: block matrices and head decay, everything else does not
    std::vector<int64_t> starts;
    std::vector<uint8_t> flags;
    const auto add = [&](int64_t start, bool decay) {
        if (!flags.empty() && flags.back() == uint8_t(decay))
            return;
        starts.push_back(start);
        flags.push_back(uint8_t(decay));
    };
    const TgParameterLayout &p = e->layout;
    add(p.embedding, false);
    for (int l = 0; l < e->config.base.depth; ++l) {
        const TgLayerParameters &b = p.layers[l];
        add(b.ln1_g, false);
        add(b.qkv, true);
        add(b.ln2_g, false);
        add(b.mlp_up, true);
    }
    add(p.lnf_g, false);
    add(p.head, true);
    e->segments = int(starts.size());
    e->allocate(e->segment_starts, starts.size(), false);
    e->allocate(e->segment_flags, flags.size(), false);
    e->upload(e->segment_starts, starts.data(), starts.size());
    e->upload(e->segment_flags, flags.data(), flags.size());
    e->sync(); // the host vectors go out of scope
}

// What the backward pass of the wide model works in.  keep: the output gradients of every block, for one launch of all
// weight gradients; otherwise one set that the blocks share.
void build_backward(Engine *e, bool keep) {
    const Config &c = e->config.base;
    const size_t M = size_t(e->tokens()), d = size_t(e->config.d_model), F = size_t(e->config.ffn), V = size_t(e->config.vocab);
    size_t need = std::max(tgk_attn_bwd_workspace(c.batch, e->config.heads, c.context), tgk_layernorm_bwd_workspace(int(M), int(d)));
    for (Slot &slot : e->slots) {
        slot.g_x.assign(c.depth + 1, nullptr);
        slot.g_mid.assign(c.depth, nullptr), slot.g_u.assign(c.depth, nullptr), slot.g_qkv.assign(c.depth, nullptr);
        slot.norms = nullptr;
        const auto allocate = [&](std::vector<bf16_t *> &buffers, size_t n) {
            for (bf16_t *&buffer : buffers)
                if (keep || &buffer == &buffers[0])
                    e->allocate(buffer, n, false);
                else
                    buffer = buffers[0];
        };
        allocate(slot.g_x, M * d);
        allocate(slot.g_mid, M * d);
        allocate(slot.g_u, M * F);
        allocate(slot.g_qkv, M * 3 * d);
        if (keep)
            e->allocate(slot.onehot, M * V, false);
        else
            slot.onehot = slot.logits; // the head's launch has read them
        float *g = slot.gradient;
        std::vector<TgkWgradJob> &jobs = slot.wgrad_jobs;
        jobs.clear();
        for (int l = 0; l < c.depth; ++l) {
            const TgLayerParameters &p = e->layout.layers[l];
            const LayerBuffers &b = slot.layers[l];
            const int D = int(d), U = int(F);
            jobs.push_back({D, U, slot.g_x[l + 1], D, b.a, U, g + p.mlp_down, U});
            jobs.push_back({U, D, slot.g_u[l], U, b.n2, D, g + p.mlp_up, D});
            jobs.push_back({D, D, slot.g_mid[l], D, b.o, D, g + p.attn_out, D});
            jobs.push_back({3 * D, D, slot.g_qkv[l], 3 * D, b.n1, D, g + p.qkv, D});
        }
        jobs.push_back({int(V), int(d), slot.logits, int(V), slot.nf, int(d), g + e->layout.head, int(d)});
        jobs.push_back({int(V), int(d), slot.onehot, int(V), slot.g_x[0], int(d), g + e->layout.embedding, int(d)});
        slot.wgrads.clear();
        if (keep) {
            slot.wgrads.push_back({0, int(jobs.size()), nullptr});
        } else {
            for (int l = 0; l < c.depth; ++l)
                slot.wgrads.push_back({4 * l, 4, nullptr});
            slot.wgrads.push_back({4 * c.depth, 1, nullptr});
            slot.wgrads.push_back({4 * c.depth + 1, 1, nullptr});
        }
        for (Slot::WgradLaunch &part : slot.wgrads) {
            const TgkWgradJob *list = jobs.data() + part.first;
            const size_t table_bytes = wgrad_list_table_bytes(int(M), part.count, list, ListUnit);
            if (!table_bytes)
                throw std::runtime_error("engine: weight gradients do not fit one list");
            uint8_t *table = nullptr;
            e->allocate(table, table_bytes, false);
            part.table = table;
            wgrad_list_prepare(int(M), part.count, list, ListUnit, table, table_bytes);
            need = std::max(need, wgrad_list_workspace(int(M), part.count, list, ListUnit));
        }
        if (!keep)
            continue; // the optimizer step takes the norm of the whole gradient itself
        // the tensors no matrix product writes, in ranges of 8192 elements (more where a long context would make
        // too many of them); with the matrices they must cover the flat gradient exactly
        struct Range {
            int64_t start, length;
        };
        std::vector<Range> ranges;
        const int64_t range = std::max<int64_t>(8192, (int64_t(c.context) * int64_t(d) / 1024 + 3) / 4 * 4);
        int64_t covered = 2 * int64_t(V) * d; // the head and the token table
        const auto cover = [&](int64_t start, int64_t length) {
            covered += length;
            for (int64_t at = 0; at < length; at += range)
                ranges.push_back({start + at, std::min<int64_t>(range, length - at)});
        };
        cover(e->layout.positions, int64_t(c.context) * d);
        for (int l = 0; l < c.depth; ++l) {
            const TgLayerParameters &p = e->layout.layers[l];
            cover(p.ln1_g, d), cover(p.ln1_b, d), cover(p.ln2_g, d), cover(p.ln2_b, d);
            covered += 4 * int64_t(d) * d + 2 * int64_t(F) * d;
        }
        cover(e->layout.lnf_g, d), cover(e->layout.lnf_b, d);
        if (covered != e->layout.count)
            throw std::runtime_error("engine: gradient norm ranges do not cover the parameters");
        slot.list_norms = wgrad_list_sumsq_count(int(M), int(slot.wgrad_jobs.size()), slot.wgrad_jobs.data(), ListUnit);
        slot.range_norms = int(ranges.size());
        if (slot.list_norms <= 0 || slot.list_norms + slot.range_norms > 4096)
            throw std::runtime_error("engine: too many gradient norm partials");
        e->allocate(slot.norms, size_t(slot.list_norms + slot.range_norms), false);
        uint8_t *device_ranges = nullptr;
        e->allocate(device_ranges, ranges.size() * sizeof(Range), false);
        check_hip(hipMemcpy(device_ranges, ranges.data(), ranges.size() * sizeof(Range), hipMemcpyHostToDevice),
                  "norm ranges: ");
        slot.norm_ranges = device_ranges;
    }
    e->workspace_bytes = need;
    const int norms = 2 * c.depth + 1;
    const size_t ln_stride = tgk_layernorm_bwd_workspace(int(M), int(d));
    for (Slot &slot : e->slots) {
        uint8_t *ws = nullptr;
        e->allocate(ws, need, false);
        slot.workspace = ws;
        e->allocate(slot.ln_partials, size_t(norms) * ln_stride, false);
        std::vector<float *> targets(size_t(2 * norms));
        targets[0] = slot.gradient + e->layout.lnf_g, targets[1] = slot.gradient + e->layout.lnf_b;
        for (int l = 0; l < c.depth; ++l) {
            const TgLayerParameters &p = e->layout.layers[l];
            targets[size_t(2 * (1 + 2 * l))] = slot.gradient + p.ln2_g, targets[size_t(2 * (1 + 2 * l) + 1)] = slot.gradient + p.ln2_b;
            targets[size_t(2 * (2 + 2 * l))] = slot.gradient + p.ln1_g, targets[size_t(2 * (2 + 2 * l) + 1)] = slot.gradient + p.ln1_b;
        }
        uint8_t *table = nullptr;
        e->allocate(table, targets.size() * sizeof(float *), false);
        check_hip(hipMemcpy(table, targets.data(), targets.size() * sizeof(float *), hipMemcpyHostToDevice));
        slot.ln_targets = table;
    }
}

} // namespace

// cuda/runtime.cu:62-155: the reference's own width-16 network (config.h:4)
TG_API Engine *tg_create(const Config *c) {
    Engine *e = nullptr;
    try {
        if (!c)
            throw std::runtime_error("Missing configuration");
        if ((c->context != 4 && c->context != 8) || (c->depth != 4 && c->depth != 8) || c->batch < 4 ||
            c->batch * c->context % 16)
            throw std::runtime_error("Supported: depth 4/8, context 4/8, batch at least 4 with "
                                     "batch*context divisible by 16");
        if (c->inflight < 1 || c->inflight > MaxInFlight)
            throw std::runtime_error("inflight must be 1.." + std::to_string(MaxInFlight));
        if (c->inflight > 1 && c->blocks)
            throw std::runtime_error("model.blocks applies to synchronous training only");
        if (c->ns_steps < 1 || c->ns_steps > 10)
            throw std::runtime_error("ns_steps must be 1..10");
        int devices = 0;
        check_hip(hipGetDeviceCount(&devices), "device query: ");
        if (c->device < 0 || c->device >= devices)
            throw std::runtime_error("No such device");
        check_hip(hipSetDevice(c->device));
        hipDeviceProp_t prop{};
        check_hip(hipGetDeviceProperties(&prop, c->device));
        if (std::strncmp(prop.gcnArchName, "gfx950", 6) != 0)
            throw std::runtime_error(std::string("Requires an MI355X-class device (gfx950), found ") +
                                     prop.gcnArchName);
        e = new Engine;
        e->width16 = true;
        e->config.base = *c;
        e->config.d_model = 16, e->config.heads = 4, e->config.vocab = 256, e->config.ffn = 48;
        e->config.ln_eps = 1e-6f;
        e->layout.count = tgk_w16_parameter_count(c->depth);
        e->compute_units = prop.multiProcessorCount;
        build_streams(e, c->inflight);
        const size_t P = size_t(e->layout.count);
        build_slots(e, c->inflight, false);
        e->allocate(e->momentum, P);
        e->allocate(e->variance, P);
        e->allocate(e->norm_partials, NormPartials);
        e->allocate(e->loss_history, size_t(HistoryRows) * c->context);
        e->allocate(e->batch_means, size_t(c->context));
        e->workspace_bytes = tgk_w16_workspace(c->depth, c->batch, c->context);
        for (Slot &slot : e->slots) {
            uint8_t *ws = nullptr;
            e->allocate(ws, e->workspace_bytes, false);
            slot.workspace = ws;
            slot.list_norms = w16_norm_count(c->depth);
            e->allocate(slot.norms, size_t(slot.list_norms * w16_norm_parts()));
        }
        e->sync();
        return e;
    } catch (const std::exception &error) {
        tg_last_error = error.what();
        delete e;
        return nullptr;
    }
}

TG_API Engine *tg_create_ex(const TgModelConfig *model) {
    Engine *e = nullptr;
    try {
        if (!model)
            throw std::runtime_error("Missing configuration");
        validate(*model);
        int devices = 0;
        check_hip(hipGetDeviceCount(&devices), "device query: ");
        if (model->base.device < 0 || model->base.device >= devices)
            throw std::runtime_error("No such device");
        check_hip(hipSetDevice(model->base.device));
        hipDeviceProp_t prop{};
        check_hip(hipGetDeviceProperties(&prop, model->base.device));
        if (std::strncmp(prop.gcnArchName, "gfx950", 6) != 0)
            throw std::runtime_error(std::string("Requires an MI355X-class device (gfx950), found ") +
                                     prop.gcnArchName);
        e = new Engine;
        e->config = *model;
        e->layout = tg_parameter_layout(model);
        e->compute_units = prop.multiProcessorCount;
        if (e->layout.count > INT_MAX)
            throw std::runtime_error("Parameter count exceeds signed 32-bit indexing");
        const Config &c = model->base;
        build_streams(e, c.inflight);
        const size_t P = size_t(e->layout.count), M = size_t(e->tokens()), d = size_t(model->d_model);
        const size_t F = size_t(model->ffn), V = size_t(model->vocab);
        build_slots(e, c.inflight, true);
        e->allocate(e->momentum, P);
        e->allocate(e->variance, P);
        e->allocate(e->norm_partials, NormPartials);
        e->allocate(e->loss_history, size_t(HistoryRows) * c.context);
        e->allocate(e->batch_means, size_t(c.context));
        build_segments(e);
        build_transpose_jobs(e);
        for (Slot &slot : e->slots) {
            slot.x.resize(c.depth + 1);
            slot.layers.resize(c.depth);
            for (int l = 0; l <= c.depth; ++l)
                e->allocate(slot.x[l], M * d, false);
            for (int l = 0; l < c.depth; ++l) {
                LayerBuffers &b = slot.layers[l];
                e->allocate(b.n1, M * d, false);
                e->allocate(b.qkv, M * 3 * d, false);
                e->allocate(b.o, M * d, false);
                e->allocate(b.lse, size_t(c.batch) * model->heads * c.context, false);
                e->allocate(b.mid, M * d, false);
                e->allocate(b.n2, M * d, false);
                e->allocate(b.u, M * F, false);
                e->allocate(b.a, M * F, false);
            }
            e->allocate(slot.nf, M * d, false);
            e->allocate(slot.logits, M * V, false);
            e->allocate(slot.t1, M * d, false);
        }
        // Every block's output gradients are kept where that leaves room for tg_batch's logits and 256 MiB of data.  It
        // takes 18 * tokens * d_model bytes a block more than one set for all of them (ffn = 4 d_model), a third of an engine.
        const size_t allocations = e->allocations.size(), bytes = e->allocated_bytes;
        bool kept = false;
        try {
            build_backward(e, true);
            size_t free = 0, total = 0;
            check_hip(hipMemGetInfo(&free, &total));
            kept = free >= M * V * sizeof(float) + (size_t(256) << 20);
        } catch (const std::exception &) {
            (void)hipGetLastError(); // the refused allocation is no later launch's error
        }
        if (!kept) {
            e->release_after(allocations, bytes);
            build_backward(e, false);
        }
        e->sync();
        return e;
    } catch (const std::exception &error) {
        tg_last_error = error.what();
        delete e;
        return nullptr;
    }
}

TG_API void tg_destroy(Engine *e) {
    delete e;
}
TG_API int tg_parameter_count(Engine *e) {
    return int(e->layout.count);
}
TG_API int tg_blocks(Engine *e) {
    return e->compute_units;
}
TG_API int tg_shared_bytes(Engine *) {
    return 3 * (128 + 192) * 64 + 4 * 4096; // the 128x192 GEMM: three 32-k stages plus the epilogue's fp32 staging tiles
}
TG_API int tg_synchronize(Engine *e) {
    return guarded([&] {
        e->use_device();
        e->sync();
    });
}
TG_API int tg_memory(Engine *e, double *used_gb) {
    return guarded([&] {
        if (!used_gb)
            throw std::runtime_error("Missing memory output");
        *used_gb = double(e->allocated_bytes) / (1024.0 * 1024.0 * 1024.0);
    });
}

// cuda/engine_state.cu:7-35
TG_API int tg_set_weights(Engine *e, const float *weights) {
    return guarded([&] {
        if (!weights)
            throw std::runtime_error("Missing weights");
        e->use_device();
        const size_t n = size_t(e->layout.count);
        std::vector<uint16_t> high(n), low(n);
        for (size_t i = 0; i < n; ++i) {
            uint32_t bits;
            std::memcpy(&bits, weights + i, 4);
            high[i] = uint16_t(bits >> 16);
            low[i] = uint16_t(bits);
        }
        e->sync(); // nothing may still read the version that is overwritten
        e->step = 0;
        e->floor = 0, e->shared_end = 0, e->shared_recorded = false;
        e->total_staleness = 0, e->max_staleness = 0;
        Version &v = e->current();
        e->upload(v.hi, high.data(), n);
        e->upload(v.lo, low.data(), n);
        check_hip(hipMemsetAsync(e->momentum, 0, n * 4, e->stream));
        check_hip(hipMemsetAsync(e->variance, 0, n * 4, e->stream));
        e->refresh_transposed(v);
        e->sync();
    });
}
// cuda/engine_state.cu:36-55
TG_API int tg_get_weights(Engine *e, float *weights) {
    return guarded([&] {
        if (!weights)
            throw std::runtime_error("Missing weights output");
        e->use_device();
        e->sync();
        e->download({{weights, size_t(e->layout.count) * 4, nullptr, e->current().hi, e->current().lo}});
    });
}
TG_API int tg_get_optimizer_state(Engine *e, float *momentum, float *variance, uint64_t *step) {
    return guarded([&] {
        if (!momentum || !variance || !step)
            throw std::runtime_error("Missing optimizer state output");
        e->use_device();
        e->sync();
        const size_t bytes = size_t(e->layout.count) * 4;
        e->download({{momentum, bytes, e->momentum}, {variance, bytes, e->variance}});
        *step = e->step;
    });
}
TG_API int tg_set_optimizer_state(Engine *e, const float *momentum, const float *variance, uint64_t step) {
    return guarded([&] {
        if (!momentum || !variance)
            throw std::runtime_error("Missing optimizer state input");
        e->use_device();
        e->sync();
        // the weights keep their values but become version `step`: move them to that place of the ring
        Version &from = e->current();
        Version &to = e->versions[step % e->versions.size()];
        if (&from != &to) {
            const size_t bytes = size_t(e->layout.count) * 2;
            check_hip(hipMemcpyAsync(to.hi, from.hi, bytes, hipMemcpyDeviceToDevice, e->stream));
            check_hip(hipMemcpyAsync(to.lo, from.lo, bytes, hipMemcpyDeviceToDevice, e->stream));
            if (to.t)
                check_hip(hipMemcpyAsync(to.t, from.t, bytes, hipMemcpyDeviceToDevice, e->stream));
        }
        e->upload(e->momentum, momentum, size_t(e->layout.count));
        e->upload(e->variance, variance, size_t(e->layout.count));
        e->step = step;
        e->floor = step, e->shared_end = step, e->shared_recorded = false;
        e->sync();
    });
}

TG_API int tg_onecycle_point(const OneCycle *schedule, int step, StepRates *rates) {
    return guarded([&] {
        if (!schedule || !rates)
            throw std::runtime_error("Missing schedule or output");
        *rates = onecycle_point(*schedule, step);
    });
}
// cuda/runtime.cu:42-61; the table stays on the host because the host issues every optimizer launch
TG_API int tg_set_onecycle(Engine *e, const OneCycle *schedule) {
    return guarded([&] {
        if (!schedule)
            throw std::runtime_error("Missing schedule");
        if (!e->schedule.empty() || e->step)
            throw std::runtime_error("Set OneCycle once, before training");
        onecycle_point(*schedule, 0); // validate before allocating
        std::vector<StepRates> rates(size_t(schedule->total_steps));
        for (int step = 0; step < schedule->total_steps; ++step)
            rates[size_t(step)] = onecycle_point(*schedule, step);
        e->schedule = std::move(rates);
    });
}

// cuda/runtime.cu:190-206
TG_API int tg_set_data(Engine *e, const uint8_t *bytes, int64_t size) {
    return guarded([&] {
        e->use_device();
        const int64_t low = std::max(8, e->config.base.context);
        if (!bytes || size <= low)
            throw std::runtime_error("Dataset needs at least " + std::to_string(low + 1) + " bytes");
        if (e->data)
            throw std::runtime_error("Dataset already loaded");
        e->allocate(e->data, size_t(size), false);
        e->data_size = size;
        e->upload(e->data, bytes, size_t(size));
        e->sync();
    });
}

// cuda/runtime.cu:213-242 with the step loop of cuda/trainer.cuh:109-124 unrolled into launches
TG_API int tg_train(Engine *e, int steps) {
    return guarded([&] {
        if (!e->data || steps < 1 || steps > MaxLaunchSteps)
            throw std::runtime_error("Load data first; each invocation permits 1.." +
                                     std::to_string(MaxLaunchSteps) + " steps");
        if (e->step + uint64_t(steps) > uint64_t(INT_MAX))
            throw std::runtime_error("Training step count exceeds signed 32-bit indexing");
        if (!e->schedule.empty() && e->step + uint64_t(steps) > e->schedule.size())
            throw std::runtime_error("Training would exceed the OneCycle schedule");
        e->use_device();
        e->version_trace.assign(size_t(steps), 0);
        e->train(e->step, steps, e->version_trace.data());
        e->last_train_steps = steps, e->last_train_first = e->step;
        e->step += uint64_t(steps);
    });
}
// cuda/engine_state.cu:76-92
TG_API int tg_get_training_losses(Engine *e, float *losses, int count) {
    return guarded([&] {
        if (!losses && count)
            throw std::runtime_error("Missing training loss output");
        if (count < 0 || count > e->last_train_steps)
            throw std::runtime_error("Training loss count exceeds the last launch");
        e->use_device();
        e->sync(); // the rows are written on the slots' streams
        const uint64_t first = e->last_train_first;
        const size_t row = size_t(e->config.base.context) * 4, together = std::min<size_t>(count, HistoryRows - first % HistoryRows);
        e->download({{losses, together * row, e->history_row(first)},
                     {losses + together * row / 4, (size_t(count) - together) * row, e->loss_history}});
    });
}
// cuda/runtime.cu:243-262: the weight version each step of the last tg_train read (a synchronous engine
// trains step s on version s)
TG_API int tg_training_versions(Engine *e, int *out, int count) {
    return guarded([&] {
        if (count < 0 || count > e->last_train_steps || (!out && count))
            throw std::runtime_error("Version trace exceeds last training launch");
        for (int i = 0; i < count; ++i)
            out[i] = e->version_trace[size_t(i)];
    });
}
// cuda/runtime.cu:263-278
TG_API int tg_pipeline_stats(Engine *e, double *mean, int *maximum) {
    return guarded([&] {
        if (!mean || !maximum)
            throw std::runtime_error("Missing pipeline statistics output");
        *mean = e->step ? double(e->total_staleness) / double(e->step) : 0;
        *maximum = e->max_staleness;
    });
}

// cuda/runtime.cu:291-320
TG_API int tg_batch(Engine *e, const uint8_t *x, const uint8_t *y, float *logits, float *gradient,
                    float *loss) {
    return guarded([&] {
        if (!x || !y || !logits || !loss)
            throw std::runtime_error("Missing batch input or output");
        e->use_device();
        const size_t M = size_t(e->tokens()), V = size_t(e->config.vocab);
        if (!e->logits_f32)
            e->allocate(e->logits_f32, M * V, false);
        e->sync_slots(); // fixed batches run on slot 0, the engine's stream, with the newest weights, after everything in flight
        Slot &slot = e->slots[0];
        check_hip(hipMemcpyAsync(slot.input, x, M, hipMemcpyHostToDevice, slot.stream));
        check_hip(hipMemcpyAsync(slot.target, y, M, hipMemcpyHostToDevice, slot.stream));
        e->forward(slot, e->current(), gradient != nullptr, e->logits_f32, e->config.base.batch);
        // with per-position means in double (cuda/runtime.cu:279-290)
        const Config &c = e->config.base;
        if (gradient)
            e->backward(slot, e->current(), e->batch_means);
        else
            ok(tgk_position_means(slot.stream, slot.token_losses, c.batch, c.context, e->batch_means));
        std::vector<ReadbackPiece> pieces = {{logits, M * V * 4, e->logits_f32}, {loss, size_t(c.context) * 4, e->batch_means}};
        if (gradient)
            pieces.push_back({gradient, size_t(e->layout.count) * 4, slot.gradient});
        e->download(pieces);
    });
}
// cuda/runtime.cu:322-351
TG_API int tg_predict(Engine *e, const uint8_t *context, float *logits) {
    return guarded([&] {
        if (!context || !logits)
            throw std::runtime_error("Missing prediction input or output");
        e->use_device();
        const Config &c = e->config.base;
        const size_t M = size_t(e->tokens()), V = size_t(e->config.vocab);
        if (!e->logits_f32)
            e->allocate(e->logits_f32, M * V, false);
        e->sync_slots();
        // Sequences do not see each other: one of them is enough.  (cuda/runtime.cu:322-351 fills the batch with copies.)
        // The wide model computes the last position's logits alone; the targets only feed losses that nobody reads.
        Slot &slot = e->slots[0];
        check_hip(hipMemcpyAsync(slot.input, context, size_t(c.context), hipMemcpyHostToDevice, slot.stream));
        e->forward(slot, e->current(), false, e->logits_f32, 1, !e->width16);
        e->download({{logits, V * 4, e->logits_f32 + (e->width16 ? size_t(c.context - 1) * V : 0)}});
    });
}
// cuda/runtime.cu:352-371
TG_API int tg_optimizer_test(Engine *e, const float *gradient, int steps) {
    return guarded([&] {
        if (!gradient)
            throw std::runtime_error("Missing gradient");
        if (e->slots.size() > 1)
            throw std::runtime_error("Optimizer oracle requires synchronous configuration");
        if (steps < 1 || steps > 64)
            throw std::runtime_error("steps must be 1..64");
        if (!e->schedule.empty() && e->step + uint64_t(steps) > e->schedule.size())
            throw std::runtime_error("Optimizer test would exceed the OneCycle schedule");
        e->use_device();
        e->upload(e->slots[0].gradient, gradient, size_t(e->layout.count));
        for (int i = 0; i < steps; ++i)
            e->optimize(e->stream, e->step + uint64_t(i), e->slots[0].gradient, e->versions[0], e->versions[0]);
        e->step += uint64_t(steps);
        e->sync();
    });
}

// Not in the reference.  One training step exactly like tg_train(engine, 1), with a HIP event pair
// around every operator launch on the engine's stream; returns the summed milliseconds and the
// number of launches per TG_CLASS_*.  Synchronises.
TG_API int tg_profile_step(Engine *e, float *class_ms, int *class_launches, int classes) {
    return guarded([&] {
        if (!class_ms || !class_launches || classes < TG_CLASSES)
            throw std::runtime_error("tg_profile_step needs room for TG_CLASSES entries");
        if (!e->data)
            throw std::runtime_error("Load data first");
        if (e->slots.size() > 1)
            throw std::runtime_error("tg_profile_step requires synchronous configuration (inflight 1)");
        if (!e->schedule.empty() && e->step + 1 > e->schedule.size())
            throw std::runtime_error("Training would exceed the OneCycle schedule");
        e->use_device();
        e->version_trace.assign(1, 0);
        e->profiling = true;
        try {
            e->train(e->step, 1, e->version_trace.data());
        } catch (...) {
            e->profiling = false;
            throw;
        }
        e->profiling = false;
        e->last_train_steps = 1, e->last_train_first = e->step;
        e->step += 1;
        e->sync();
        std::fill(class_ms, class_ms + classes, 0.f);
        std::fill(class_launches, class_launches + classes, 0);
        for (Engine::Span &span : e->spans) {
            float ms = 0.f;
            check_hip(hipEventElapsedTime(&ms, span.start, span.stop));
            class_ms[span.cls] += ms;
            class_launches[span.cls] += 1;
            e->event_pool.push_back(span.start);
            e->event_pool.push_back(span.stop);
        }
        e->spans.clear();
    });
}
