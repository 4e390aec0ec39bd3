#include "unet.h"

#include <cmath>
#include <cstring>
#include <random>
#include <stdexcept>

#include "domain.h"

namespace artss {

namespace {

struct Spec {
    int ci, co, level;
};
// layer order of the parameter vector
const Spec kLayers[] = {{2, 16, 0},  {16, 16, 0}, {16, 32, 1}, {32, 64, 2}, {64, 64, 3},
                        {64, 64, 2}, {64, 32, 1}, {32, 16, 0}, {16, 1, 0}};
enum { L_IN, L_E0, L_E1, L_E2, L_E3, L_D2, L_D1, L_D0, L_OUT, NLAYERS };
// the layers that read a nearest-upsampled input
inline bool upsampling(size_t layer) { return layer == L_D2 || layer == L_D1 || layer == L_D0; }

template <typename T>
T *dalloc(size_t n, std::vector<void *> *owner = nullptr) {
    T *p = nullptr;
    ARTSS_HIP(hipMalloc(&p, sizeof(T) * (n ? n : 1)));
    ARTSS_HIP(hipMemset(p, 0, sizeof(T) * (n ? n : 1)));
    if (owner) owner->push_back(p);
    return p;
}

}  // namespace

size_t UNet::param_count() {
    size_t n = 0;
    for (const Spec &s : kLayers) n += 27 * s.ci * s.co + s.co;
    return n;
}

UNet::UNet(hipStream_t stream, unsigned long long seed) : m_s(stream) {
    std::mt19937_64 rng(seed);
    std::normal_distribution<double> nd(0.0, 1.0);
    const size_t n = param_count();
    m_params = dalloc<float>(n);
    m_grads = dalloc<float>(n + 1);
    m_m = dalloc<float>(n);
    m_v = dalloc<float>(n);
    std::vector<float> host(n, 0.f);
    size_t off = 0;
    for (const Spec &s : kLayers) {
        Layer L;
        L.ci = s.ci;
        L.co = s.co;
        L.level = s.level;
        const size_t nw = 27 * static_cast<size_t>(s.ci) * s.co;
        L.w = off;
        L.b = off + nw;
        if (s.ci >= 16 && s.co >= 16) {
            const bool up = upsampling(m_layers.size());
            const size_t pair = static_cast<size_t>(s.ci) * s.co;
            L.fwd = dalloc<uint16_t>((up ? 64 : 27) * pair);
            L.bwd = dalloc<uint16_t>((up ? 192 : 27) * pair);
        }
        // He initialisation; the output layer starts at zero, so an untrained
        // network predicts no correction
        const bool out_layer = m_layers.size() + 1 == sizeof(kLayers) / sizeof(kLayers[0]);
        const double std_ = out_layer ? 0.0 : std::sqrt(2.0 / (27.0 * s.ci));
        for (size_t q = 0; q < nw; q++) host[off + q] = static_cast<float>(std_ * nd(rng));
        off += nw + static_cast<size_t>(s.co);
        m_layers.push_back(L);
    }
    ARTSS_HIP(hipMemcpy(m_params, host.data(), sizeof(float) * n, hipMemcpyHostToDevice));
    ARTSS_HIP(hipHostMalloc(&m_grads_host, sizeof(float) * (n + 1)));
    refresh_weights();
    ARTSS_HIP(hipStreamSynchronize(m_s));
}

UNet::~UNet() {
    (void)hipStreamSynchronize(m_s);
    free_buffers();
    for (Layer &L : m_layers)
        for (void *p : {static_cast<void *>(L.fwd), static_cast<void *>(L.bwd)})
            if (p) (void)hipFree(p);
    for (float *p : {m_params, m_grads, m_m, m_v}) (void)hipFree(p);
    (void)hipHostFree(m_grads_host);
}

// the BF16 copies follow the FP32 weights
void UNet::refresh_weights() {
    nn::WeightJobs jobs{};
    for (size_t q = 0; q < m_layers.size(); q++) {
        const Layer &L = m_layers[q];
        if (L.fwd) jobs.job[jobs.count++] = nn::WeightJob{m_params + L.w, L.ci, L.co, upsampling(q) ? 1 : 0, L.fwd, L.bwd};
    }
    nn::weights_bf16(m_s, jobs);
}

void UNet::set_params(const float *host) {
    const size_t n = param_count();
    ARTSS_HIP(hipStreamSynchronize(m_s));
    ARTSS_HIP(hipMemcpy(m_params, host, sizeof(float) * n, hipMemcpyHostToDevice));
    ARTSS_HIP(hipMemset(m_m, 0, sizeof(float) * n));
    ARTSS_HIP(hipMemset(m_v, 0, sizeof(float) * n));
    refresh_weights();
    m_adam_t = 0;
    ARTSS_HIP(hipStreamSynchronize(m_s));
}

void UNet::get_params(float *host) const {
    ARTSS_HIP(hipStreamSynchronize(m_s));
    ARTSS_HIP(hipMemcpy(host, m_params, sizeof(float) * param_count(), hipMemcpyDeviceToHost));
}

void UNet::free_buffers() {
    for (void *p : m_buffers) (void)hipFree(p);
    m_buffers.clear();
    m_backward = false;
    m_X = m_Y = m_Z = 0;
}

void UNet::ensure(int X, int Y, int Z) {
    if (X == m_X && Y == m_Y && Z == m_Z) return;
    if (X <= 0 || Y <= 0 || Z <= 0 || X % 8 || Y % 8 || Z % 8)
        throw std::invalid_argument("U-Net volume sides must be positive multiples of 8");
    ARTSS_HIP(hipStreamSynchronize(m_s));
    free_buffers();
    const size_t V0 = static_cast<size_t>(X) * Y * Z, V1 = V0 / 8, V2 = V1 / 8, V3 = V2 / 8;
    auto b16 = [&](size_t n) { return dalloc<uint16_t>(n, &m_buffers); };
    h0 = b16(V0 * 16);
    e0 = b16(V0 * 16);
    p1 = b16(V1 * 16);
    e1 = b16(V1 * 32);
    p2 = b16(V2 * 32);
    e2 = b16(V2 * 64);
    p3 = b16(V3 * 64);
    e3 = b16(V3 * 64);
    d2 = b16(V2 * 64);
    d1 = b16(V1 * 32);
    d0 = b16(V0 * 16);
    y = dalloc<float>(V0, &m_buffers);
    m_X = X;
    m_Y = Y;
    m_Z = Z;
}

namespace {
// the partial-row buffers of one backward pass, in the order they are used:
// counts the floats when there is no buffer yet, hands out rows when there is
struct Rows {
    float *base;
    size_t used = 0;
    nn::SumJobs jobs{};
    float *rows(int count, int stride) {
        float *p = base ? base + used : nullptr;
        used += static_cast<size_t>(count) * stride;
        return p;
    }
    void sum(const float *part, int count, int stride, int n, float scale, float *out) {
        if (jobs.count >= nn::kMaxSumJobs) throw std::logic_error("more sums than a launch holds");
        jobs.job[jobs.count++] = nn::SumJob{part, count, stride, n, scale, out};
    }
};
}  // namespace

void UNet::ensure_backward() {
    if (m_backward) return;
    const size_t V0 = static_cast<size_t>(m_X) * m_Y * m_Z, V1 = V0 / 8, V2 = V1 / 8, V3 = V2 / 8;
    auto b16 = [&](size_t n) { return dalloc<uint16_t>(n, &m_buffers); };
    auto f32 = [&](size_t n) { return dalloc<float>(n, &m_buffers); };
    c2 = b16(V2 * 64);
    c1 = b16(V1 * 32);
    c0 = b16(V0 * 16);
    gy = f32(V0);
    gs[0] = f32(V0 * 16);
    gs[1] = f32(V1 * 32);
    gs[2] = f32(V2 * 64);
    gp[0] = f32(V1 * 16);
    gp[1] = f32(V2 * 32);
    gp[2] = f32(V3 * 64);
    gh = f32(V0 * 16);
    gm[0] = b16(V0 * 16);
    gm[1] = b16(V1 * 32);
    gm[2] = b16(V2 * 64);
    gm[3] = b16(V3 * 64);
    m_part = nullptr;
    m_backward = true;
}

void UNet::run_forward(const float *x, bool keep_pre) {
    const nn::Dims D0{m_X, m_Y, m_Z}, D1{m_X / 2, m_Y / 2, m_Z / 2}, D2{m_X / 4, m_Y / 4, m_Z / 4},
        D3{m_X / 8, m_Y / 8, m_Z / 8};
    const Layer *L = m_layers.data();
    nn::conv_in(m_s, D0, x, W(L_IN), B(L_IN), h0);
    nn::conv_fwd(m_s, 16, 16, false, D0, h0, L[L_E0].fwd, B(L_E0), e0, nullptr, nullptr, true);
    nn::down(m_s, 16, D1, e0, p1);
    nn::conv_fwd(m_s, 16, 32, false, D1, p1, L[L_E1].fwd, B(L_E1), e1, nullptr, nullptr, true);
    nn::down(m_s, 32, D2, e1, p2);
    nn::conv_fwd(m_s, 32, 64, false, D2, p2, L[L_E2].fwd, B(L_E2), e2, nullptr, nullptr, true);
    nn::down(m_s, 64, D3, e2, p3);
    nn::conv_fwd(m_s, 64, 64, false, D3, p3, L[L_E3].fwd, B(L_E3), e3, nullptr, nullptr, true);
    nn::conv_fwd(m_s, 64, 64, true, D2, e3, L[L_D2].fwd, B(L_D2), d2, keep_pre ? c2 : nullptr, e2, true);
    nn::conv_fwd(m_s, 64, 32, true, D1, d2, L[L_D1].fwd, B(L_D1), d1, keep_pre ? c1 : nullptr, e1, true);
    nn::conv_fwd(m_s, 32, 16, true, D0, d1, L[L_D0].fwd, B(L_D0), d0, keep_pre ? c0 : nullptr, e0, true);
    nn::conv_out(m_s, D0, d0, W(L_OUT), B(L_OUT), y);
    m_x = x;
}

void UNet::forward(int X, int Y, int Z, const float *x, float *out) {
    ensure(X, Y, Z);
    run_forward(x, false);
    ARTSS_HIP(hipMemcpyAsync(out, y, sizeof(float) * static_cast<size_t>(X) * Y * Z, hipMemcpyDeviceToDevice, m_s));
    ARTSS_HIP(hipStreamSynchronize(m_s));
}

// Backward through every layer.  With m_part == nullptr only the partial
// rows are counted and allocated; every sum then runs in one launch at the
// end (nn::sum_rows).
void UNet::run_backward(const float *target) {
    const nn::Dims D0{m_X, m_Y, m_Z}, D1{m_X / 2, m_Y / 2, m_Z / 2}, D2{m_X / 4, m_Y / 4, m_Z / 4},
        D3{m_X / 8, m_Y / 8, m_Z / 8};
    const long long V0 = static_cast<long long>(m_X) * m_Y * m_Z;
    const Layer *L = m_layers.data();
    for (int pass = m_part ? 1 : 0; pass < 2; pass++) {
        const bool run = pass == 1;
        Rows R{m_part};
        auto gW = [&](int layer) { return m_grads + L[layer].w; };
        auto gb = [&](int layer) { return m_grads + L[layer].b; };
        auto wgrad = [&](int layer, bool up, nn::Dims D, const uint16_t *in, const uint16_t *g) {
            const int ci = L[layer].ci, co = L[layer].co, n = 27 * ci * co, rows = nn::wgrad_rows(ci, co, D);
            float *part = R.rows(rows, n);
            if (run) nn::conv_wgrad(m_s, ci, co, up, D, in, g, part);
            R.sum(part, rows, n, n, 1.f, gW(layer));
        };
        // the gradient at the coarse input of decoder layer `layer`, whose
        // channel sums are the bias gradient of `below`
        auto up_dgrad = [&](int layer, int below, nn::Dims Dc, const uint16_t *g, const uint16_t *act, float *gskip,
                            uint16_t *gmask) {
            const int ci = L[layer].ci, co = L[layer].co, rows = nn::up_dgrad_rows(ci, co, Dc);
            float *part = R.rows(rows, ci);
            if (run) nn::conv_up_dgrad(m_s, ci, co, Dc, g, L[layer].bwd, act, gskip, gmask, part);
            R.sum(part, rows, ci, ci, 1.f, gb(below));
        };
        auto enc = [&](int layer, nn::Dims D, const float *gskip, const float *gc, const uint16_t *act,
                       uint16_t *gmask) {
            const int c = L[layer].co;
            const int rows = nn::elementwise_rows(static_cast<long long>(D.X) * D.Y * D.Z, c / 4);
            float *part = R.rows(rows, c);
            if (run) nn::enc_grad(m_s, c, D, gskip, gc, act, gmask, part);
            R.sum(part, rows, c, c, 1.f, gb(layer));
        };
        // loss and output layer
        {
            const int rows = nn::elementwise_rows(V0, 1);
            float *part = R.rows(rows, 4);
            if (run) nn::mse(m_s, V0, y, target, gy, part);
            R.sum(part, rows, 4, 1, 1.f / static_cast<float>(V0), m_grads + param_count());
            R.sum(part ? part + 1 : nullptr, rows, 4, 1, 1.f, gb(L_OUT));
            const int wrows = nn::end_wgrad_rows(D0);
            float *wpart = R.rows(wrows, 27 * 16);
            if (run) nn::conv_out_wgrad(m_s, D0, d0, gy, wpart);
            R.sum(wpart, wrows, 27 * 16, 27 * 16, 1.f, gW(L_OUT));
            const int drows = nn::end_dgrad_rows(D0);
            float *dpart = R.rows(drows, 16);
            if (run) nn::conv_out_dgrad(m_s, D0, W(L_OUT), gy, c0, gs[0], gm[0], dpart);
            R.sum(dpart, drows, 16, 16, 1.f, gb(L_D0));
        }
        // decoder: weight gradient, then the gradient at the layer's coarse input
        wgrad(L_D0, true, D0, d1, gm[0]);
        up_dgrad(L_D0, L_D1, D1, gm[0], c1, gs[1], gm[1]);
        wgrad(L_D1, true, D1, d2, gm[1]);
        up_dgrad(L_D1, L_D2, D2, gm[1], c2, gs[2], gm[2]);
        wgrad(L_D2, true, D2, e3, gm[2]);
        up_dgrad(L_D2, L_E3, D3, gm[2], e3, nullptr, gm[3]);
        // encoder, coarsest first
        wgrad(L_E3, false, D3, p3, gm[3]);
        if (run) nn::conv_dgrad(m_s, 64, 64, D3, gm[3], L[L_E3].bwd, nullptr, gp[2]);
        enc(L_E2, D2, gs[2], gp[2], e2, gm[2]);
        wgrad(L_E2, false, D2, p2, gm[2]);
        if (run) nn::conv_dgrad(m_s, 32, 64, D2, gm[2], L[L_E2].bwd, nullptr, gp[1]);
        enc(L_E1, D1, gs[1], gp[1], e1, gm[1]);
        wgrad(L_E1, false, D1, p1, gm[1]);
        if (run) nn::conv_dgrad(m_s, 16, 32, D1, gm[1], L[L_E1].bwd, nullptr, gp[0]);
        enc(L_E0, D0, gs[0], gp[0], e0, gm[0]);
        wgrad(L_E0, false, D0, h0, gm[0]);
        {
            const int rows = nn::end_wgrad_rows(D0), n = 55 * 16;
            float *part = R.rows(rows, n);
            if (run) {
                nn::conv_dgrad(m_s, 16, 16, D0, gm[0], L[L_E0].bwd, h0, gh);
                nn::conv_in_wgrad(m_s, D0, m_x, gh, part);
            }
            R.sum(part, rows, n, n, 1.f, gW(L_IN));  // W, then b, as in the parameter vector
        }
        if (run) nn::sum_rows(m_s, R.jobs);
        else m_part = dalloc<float>(R.used, &m_buffers);
    }
}

float UNet::gradients(int X, int Y, int Z, const float *x, const float *target, float *grads) {
    ensure(X, Y, Z);
    ensure_backward();
    run_forward(x, true);
    run_backward(target);
    const size_t n = param_count();
    // the loss stands behind the gradients: one copy, through pinned memory
    const size_t first = grads ? 0 : n;
    ARTSS_HIP(hipMemcpyAsync(m_grads_host + first, m_grads + first, sizeof(float) * (n + 1 - first),
                             hipMemcpyDeviceToHost, m_s));
    ARTSS_HIP(hipStreamSynchronize(m_s));
    if (grads) std::memcpy(grads, m_grads_host, sizeof(float) * n);
    return m_grads_host[n];
}

void UNet::adam_step(float lr) {
    const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
    m_adam_t++;
    const float c1 = 1.f - std::pow(b1, static_cast<float>(m_adam_t));
    const float c2 = 1.f - std::pow(b2, static_cast<float>(m_adam_t));
    nn::adam(m_s, static_cast<int>(param_count()), m_params, m_grads, m_m, m_v, lr, b1, b2, eps, c1, c2);
    refresh_weights();
}

}  // namespace artss
