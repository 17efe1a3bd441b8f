// spk_guide_api.cpp -- C ABI of the learned path-guiding proposal (include/spk.h).
//
// spica has no learned sampling; these entry points own the network's parameters and
// Adam state, evaluate it for checks against the CPU oracle, and train it on given
// batches.  Online training inside a render goes through spk_render_set_guide (spk_api.cpp).
#include <math.h>
#include <string.h>

#include <algorithm>
#include <memory>
#include <vector>

#include "spk_internal.h"
#include "spk_sampler.h"

using namespace spk;

spk::GuideBufsDev spk_guide::bufs() const {
    GuideBufsDev b;
    b.params = params.as<float>();
    b.m = m.as<float>();
    b.v = v.as<float>();
    b.wf = wf.as<uint16_t>();
    b.wb = wb.as<uint16_t>();
    b.bias = bias.as<float>();
    b.partial = partial.as<float>();
    b.psum = psum.as<float>();
    b.gnorm_part = gnorm_part.as<float>();
    b.loss_part = loss_part.as<float2>();
    b.gs = state.as<GuideState>();
    b.grid = cus;
    return b;
}

spk::TrainBufs spk_guide::train_bufs(uint32_t ncols) const {
    TrainBufs t;
    for (int k = 0; k < 3; k++) t.tb[k] = tb[k].as<float4>();
    t.act = act.as<uint16_t>();
    t.dz = dz.as<uint16_t>();
    t.ld = bcap;
    t.ncols = ncols;
    t.batch = (uint32_t)opts.batch_size;
    return t;
}

spk::AdamCfg spk_guide::adam() const {
    AdamCfg c;
    c.lr = opts.learning_rate;
    c.beta1 = opts.beta1;
    c.beta2 = opts.beta2;
    c.eps = opts.epsilon;
    return c;
}

namespace {

// Xavier-uniform weights from a counter-based hash of (seed, index); zero biases.
void init_params(uint32_t seed, std::vector<float>& th) {
    th.assign(kGParams, 0.0f);
    const int offW[5] = {kGOffW1, kGOffW2, kGOffW3, kGOffW4, kGOffW5};
    const int rows[5] = {kGHid, kGHid, kGHid, kGHid, kGOut};
    const int cols[5] = {kGEnc, kGHid, kGHid, kGHid, kGHid};
    for (int l = 0; l < 5; l++) {
        const double s = sqrt(6.0 / (rows[l] + cols[l]));
        for (int i = 0; i < rows[l] * cols[l]; i++) {
            uint32_t a = (uint32_t)(offW[l] + i), b = seed, c = 0x243f6a88u, d = 0x85a308d3u;
            pcg4d(a, b, c, d);
            const double u = (double)(a >> 8) * (1.0 / 16777216.0);
            th[offW[l] + i] = (float)((2.0 * u - 1.0) * s);
        }
    }
}

int upload_params(spk_guide* g, const float* th) {
    int rc;
    SPK_CHECK_HIP(hipMemcpyAsync(g->params.p, th, kGParams * 4, hipMemcpyHostToDevice, g->stream));
    SPK_CHECK_HIP(hipMemsetAsync(g->m.p, 0, kGParams * 4, g->stream));
    SPK_CHECK_HIP(hipMemsetAsync(g->v.p, 0, kGParams * 4, g->stream));
    SPK_CHECK_HIP(hipMemsetAsync(g->state.p, 0, sizeof(GuideState), g->stream));
    if ((rc = launch_guide_images(g->params.as<float>(), g->wf.as<uint16_t>(), g->wb.as<uint16_t>(), g->bias.as<float>(),
                                  g->stream)))
        return rc;
    SPK_CHECK_HIP(hipStreamSynchronize(g->stream));
    g->steps = 0;
    return SPK_OK;
}

int check_n(spk_guide* g, int64_t n, const char* fn) {
    if (!g || n < 0) {
        set_error("%s: bad arguments", fn);
        return SPK_ERR_INVALID;
    }
    return SPK_OK;
}

// Callers' arrays go to the device as they are (a kernel lays them out there) through one staging
// buffer that the handle keeps: packing and padding them on the host took longer than a gradient's
// kernels, and a hipMalloc and hipFree an array longer still (gradient of 2^18 samples 1.25 ms -> 0.64 ms, of
// which the upload is 0.35; 100,003 sampled directions 0.56 -> 0.29 ms).  It holds a batch, or a piece of
// kEvalPiece queries: evaluations of any size go through in pieces.
constexpr int64_t kEvalPiece = int64_t(1) << 17;

int stage_room(spk_guide* g, size_t bytes) { return g->stage.bytes >= bytes ? SPK_OK : g->stage.alloc(bytes); }

// Uploads a direct batch into the training arrays.
int upload_batch(spk_guide* g, int64_t n, const float* x, const float* dirs, const float* weight, const TrainBufs& tb) {
    const size_t N = (size_t)n;
    int rc;
    if ((rc = stage_room(g, N * 44))) return rc;
    float *dx = g->stage.as<float>(), *dd = dx + 7 * N, *dw = dd + 3 * N;
    SPK_CHECK_HIP(hipMemcpyAsync(dx, x, N * 28, hipMemcpyHostToDevice, g->stream));
    SPK_CHECK_HIP(hipMemcpyAsync(dd, dirs, N * 12, hipMemcpyHostToDevice, g->stream));
    SPK_CHECK_HIP(hipMemcpyAsync(dw, weight, N * 4, hipMemcpyHostToDevice, g->stream));
    return launch_guide_pack(dx, dd, dw, (uint32_t)n, tb, g->stream);
}

// Evaluations in pieces: mode 0 the outputs and log densities, mode 1 sampled directions and densities
// (out_raw, out_dir and out_pdf may be null where the mode does not need them).
int eval_pieces(spk_guide* g, int mode, int64_t n, const float* x, const float* aux, float* out_raw, float* out_dir,
                float* out_pdf) {
    const size_t P = (size_t)std::min(n, kEvalPiece);
    int rc;
    if ((rc = stage_room(g, P * (40 + 16 + (out_raw ? kGOut * 4 : 0))))) return rc;
    float *dx = g->stage.as<float>(), *da = dx + 7 * P, *dd = da + 3 * P, *dp = dd + 3 * P, *dr = dp + P;
    for (int64_t i0 = 0; i0 < n; i0 += kEvalPiece) {
        const size_t m = (size_t)std::min(kEvalPiece, n - i0);
        SPK_CHECK_HIP(hipMemcpyAsync(dx, x + 7 * i0, m * 28, hipMemcpyHostToDevice, g->stream));
        SPK_CHECK_HIP(hipMemcpyAsync(da, aux + 3 * i0, m * 12, hipMemcpyHostToDevice, g->stream));
        if ((rc = launch_guide_eval(mode, g->wf.as<uint16_t>(), g->bias.as<float>(), (int64_t)m, dx, da,
                                    out_raw ? dr : nullptr, dd, out_pdf ? dp : nullptr, g->cus, g->stream)))
            return rc;
        if (out_raw) SPK_CHECK_HIP(hipMemcpyAsync(out_raw + kGOut * i0, dr, m * kGOut * 4, hipMemcpyDeviceToHost, g->stream));
        if (out_dir) SPK_CHECK_HIP(hipMemcpyAsync(out_dir + 3 * i0, dd, m * 12, hipMemcpyDeviceToHost, g->stream));
        if (out_pdf) SPK_CHECK_HIP(hipMemcpyAsync(out_pdf + i0, dp, m * 4, hipMemcpyDeviceToHost, g->stream));
        SPK_CHECK_HIP(hipStreamSynchronize(g->stream));
    }
    return SPK_OK;
}

int eval_grid(int device) {
    hipDeviceProp_t prop;
    if (hipGetDeviceProperties(&prop, device) != hipSuccess) return 256;
    return prop.multiProcessorCount;
}

}  // namespace

extern "C" {

int spk_guide_opts_default(spk_guide_opts* o) {
    clear_error();
    if (!o) return SPK_ERR_INVALID;
    memset(o, 0, sizeof(*o));
    o->seed = 1;
    o->batch_size = 1 << 18;
    o->steps_per_pass = 8;
    o->train_spp = 64;
    o->learning_rate = 1.0e-2f;
    o->beta1 = 0.95f;  // C3 over twelve render seeds: 0.8 0.593, 0.9 0.602, 0.95 0.569, 0.97 0.609
    // A short second-moment memory: a record whose radiance estimate F/p is far above the rest
    // (a caustic path found by BSDF sampling) gives one step a gradient orders of magnitude
    // larger than the others.  With beta2 = 0.999 that step moves every weight by ~3 lr and
    // then holds the second moment up for hundreds of steps, so the steps after it barely move;
    // with 0.95 the spike's own step is ~0.45 lr and training recovers within ~20 steps.
    o->beta2 = 0.95f;
    o->epsilon = 1.0e-8f;
    o->guide_fraction = 0.5f;
    o->train_pass_spp = 8;
    o->glossy_min_alpha = 0.5f;
    o->guided_depth = 3;
    return SPK_OK;
}

int64_t spk_guide_num_params(void) { return kGParams; }

int spk_guide_create(int device, const spk_guide_opts* opts, spk_guide** out) {
    clear_error();
    if (!out) return SPK_ERR_INVALID;
    *out = nullptr;
    // the options first (no device needed to reject them)
    spk_guide_opts o;
    spk_guide_opts_default(&o);
    if (opts) o = *opts;
    if (o.batch_size < 64 || o.batch_size > (1 << 22) || o.batch_size % 64 != 0) {
        set_error("spk_guide_create: batch_size %d must be a multiple of 64 in [64, 2^22]", o.batch_size);
        return SPK_ERR_INVALID;
    }
    if (o.steps_per_pass < 0 || o.train_spp < 0 || o.train_pass_spp < 1 || !(o.learning_rate > 0.0f) || !(o.guide_fraction >= 0.0f) ||
        !(o.guide_fraction < 1.0f) || !(o.beta1 >= 0.0f && o.beta1 < 1.0f) || !(o.beta2 >= 0.0f && o.beta2 < 1.0f) ||
        !(o.glossy_min_alpha >= 0.0f && o.glossy_min_alpha < 1.0e30f) || o.guided_depth < 1) {
        set_error("spk_guide_create: bad options");
        return SPK_ERR_INVALID;
    }
    int ndev = 0;
    SPK_CHECK_HIP(hipGetDeviceCount(&ndev));
    if (device < 0 || device >= ndev) {
        set_error("spk_guide_create: device %d not present", device);
        return SPK_ERR_INVALID;
    }
    std::unique_ptr<spk_guide> g(new spk_guide());
    g->device = device;
    g->opts = o;
    SPK_CHECK_HIP(hipSetDevice(device));
    SPK_CHECK_HIP(hipStreamCreateWithFlags(&g->stream, hipStreamNonBlocking));
    g->bcap = (uint32_t)o.batch_size;
    g->cus = eval_grid(device);
    const size_t B = g->bcap;
    const size_t splits = (B + kGuideColsPerSplit - 1) / kGuideColsPerSplit;
    int rc;
    if ((rc = g->params.alloc(kGParams * 4)) || (rc = g->m.alloc(kGParams * 4)) || (rc = g->v.alloc(kGParams * 4)) ||
        (rc = g->wf.alloc(kGFwdSize * 2)) || (rc = g->wb.alloc(kGBwdSize * 2)) || (rc = g->bias.alloc(kGBiasSize * 4)) ||
        (rc = g->partial.alloc(splits * kGParams * 4)) || (rc = g->psum.alloc((size_t)kPsumGroups * kGParams * 4)) ||
        (rc = g->state.alloc(sizeof(GuideState))) ||
        (rc = g->grad.alloc(kGParams * 4)) || (rc = g->gnorm_part.alloc(kGnormBlocks * 4)) ||
        (rc = g->loss_part.alloc((size_t)std::max(1, g->cus) * 8)))
        return rc;
    for (int k = 0; k < 3; k++)
        if ((rc = g->tb[k].alloc(B * 16))) return rc;
    if ((rc = g->act.alloc(B * 4 * 64 * 2)) || (rc = g->dz.alloc(B * 5 * 64 * 2)))
        return rc;
    // padding of the bf16 images and biases stays zero
    SPK_CHECK_HIP(hipMemset(g->wf.p, 0, kGFwdSize * 2));
    SPK_CHECK_HIP(hipMemset(g->wb.p, 0, kGBwdSize * 2));
    SPK_CHECK_HIP(hipMemset(g->bias.p, 0, kGBiasSize * 4));
    std::vector<float> th;
    init_params(o.seed, th);
    if ((rc = upload_params(g.get(), th.data()))) return rc;
    *out = g.release();
    return SPK_OK;
}

int spk_guide_destroy(spk_guide* g) {
    clear_error();
    if (!g) return SPK_OK;
    (void)hipSetDevice(g->device);
    if (g->stream) {
        (void)hipStreamSynchronize(g->stream);
        (void)hipStreamDestroy(g->stream);
    }
    DevBuf* b[] = {&g->params, &g->m, &g->v, &g->wf, &g->wb, &g->bias, &g->partial, &g->psum, &g->state, &g->grad,
                   &g->gnorm_part, &g->loss_part, &g->tb[0], &g->tb[1], &g->tb[2], &g->act, &g->dz, &g->stage};
    for (DevBuf* x : b) x->release();
    delete g;
    return SPK_OK;
}

int spk_guide_params_get(spk_guide* g, float* out) {
    clear_error();
    if (!g || !out) return SPK_ERR_INVALID;
    SPK_CHECK_HIP(hipSetDevice(g->device));
    SPK_CHECK_HIP(hipDeviceSynchronize());
    SPK_CHECK_HIP(hipMemcpy(out, g->params.p, kGParams * 4, hipMemcpyDeviceToHost));
    return SPK_OK;
}

int spk_guide_params_set(spk_guide* g, const float* in) {
    clear_error();
    if (!g || !in) return SPK_ERR_INVALID;
    SPK_CHECK_HIP(hipSetDevice(g->device));
    SPK_CHECK_HIP(hipDeviceSynchronize());
    return upload_params(g, in);
}

int spk_guide_eval(spk_guide* g, int64_t n, const float* x, const float* dirs, float* out_raw, float* log_pdf) {
    clear_error();
    int rc;
    if ((rc = check_n(g, n, "spk_guide_eval"))) return rc;
    if (n == 0) return SPK_OK;
    if (!x || !dirs) return SPK_ERR_INVALID;
    SPK_CHECK_HIP(hipSetDevice(g->device));
    return eval_pieces(g, 0, n, x, dirs, out_raw, nullptr, log_pdf);
}

int spk_guide_sample(spk_guide* g, int64_t n, const float* x, const float* u, float* dirs, float* pdf) {
    clear_error();
    int rc;
    if ((rc = check_n(g, n, "spk_guide_sample"))) return rc;
    if (n == 0) return SPK_OK;
    if (!x || !u || !dirs) return SPK_ERR_INVALID;
    SPK_CHECK_HIP(hipSetDevice(g->device));
    return eval_pieces(g, 1, n, x, u, nullptr, dirs, pdf);
}

static int direct_steps(spk_guide* g, int64_t n, const float* x, const float* dirs, const float* weight, int32_t steps,
                        float* grad, double* loss) {
    int rc;
    if ((rc = check_n(g, n, grad ? "spk_guide_grad" : "spk_guide_train"))) return rc;
    if (n == 0 || steps <= 0) return SPK_OK;
    if (!x || !dirs || !weight || n > (int64_t)g->bcap) {
        set_error("spk_guide: n = %lld must be in [1, batch_size = %u]", (long long)n, g->bcap);
        return SPK_ERR_INVALID;
    }
    SPK_CHECK_HIP(hipSetDevice(g->device));
    const uint32_t ncols = (uint32_t)((n + 63) / 64 * 64);
    const TrainBufs tb = g->train_bufs(ncols);
    if ((rc = upload_batch(g, n, x, dirs, weight, tb))) return rc;
    for (int s = 0; s < steps; s++) {
        if ((rc = launch_guide_step(g->bufs(), tb, nullptr, g->adam(), (uint32_t)g->steps, (uint32_t)n,
                                    grad == nullptr, grad ? g->grad.as<float>() : nullptr, g->stream)))
            return rc;
        if (!grad) g->steps++;
    }
    GuideState st;
    if (grad) SPK_CHECK_HIP(hipMemcpyAsync(grad, g->grad.p, kGParams * 4, hipMemcpyDeviceToHost, g->stream));
    if (loss) SPK_CHECK_HIP(hipMemcpyAsync(&st, g->state.p, sizeof(st), hipMemcpyDeviceToHost, g->stream));
    SPK_CHECK_HIP(hipStreamSynchronize(g->stream));
    if (loss) *loss = (double)st.loss_sum / (double)n;
    return SPK_OK;
}

int spk_guide_grad(spk_guide* g, int64_t n, const float* x, const float* dirs, const float* weight, float* grad,
                   double* loss) {
    clear_error();
    if (!grad) return SPK_ERR_INVALID;
    return direct_steps(g, n, x, dirs, weight, 1, grad, loss);
}

int spk_guide_train(spk_guide* g, int64_t n, const float* x, const float* dirs, const float* weight, int32_t steps) {
    clear_error();
    return direct_steps(g, n, x, dirs, weight, steps, nullptr, nullptr);
}

int spk_guide_set_train_spp(spk_guide* g, int32_t train_spp) {
    clear_error();
    if (!g || train_spp < 0) return SPK_ERR_INVALID;
    g->opts.train_spp = train_spp;
    return SPK_OK;
}

int spk_guide_stats_get(spk_guide* g, spk_guide_stats* out) {
    clear_error();
    if (!g || !out) return SPK_ERR_INVALID;
    SPK_CHECK_HIP(hipSetDevice(g->device));
    SPK_CHECK_HIP(hipDeviceSynchronize());
    GuideState st;
    SPK_CHECK_HIP(hipMemcpy(&st, g->state.p, sizeof(st), hipMemcpyDeviceToHost));
    memset(out, 0, sizeof(*out));
    out->steps = (int64_t)st.t;
    out->last_records = (int64_t)st.n_rec;
    out->last_loss = st.b_eff ? (double)st.loss_sum / st.b_eff : 0.0;
    out->last_weight = st.b_eff ? (double)st.weight_sum / st.b_eff : 0.0;
    return SPK_OK;
}

}  // extern "C"
