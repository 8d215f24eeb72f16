// C-ABI of the warm-start network (include/plsqr_hip.h, plsqr_cnn_*): a
// 4-layer 3x3x3 convolutional network, 32 channels, bf16 weights and
// activations with FP32 accumulation on the MFMA units, trained on the GPU
// with Adam on FP32 master weights.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <mutex>
#include <string>
#include <vector>

#include "plsqr_cnn.h"
#include "plsqr_hip.h"

using namespace plsqr::cnn;

namespace {

constexpr int LAYERS = 4;
constexpr int WSZ = TAPS * C * C;      // weights of one layer
constexpr int LSZ = WSZ + C;           // weights + bias
constexpr int NPARAM = LAYERS * LSZ + 1;  // + the output gain (last entry, not trained)
constexpr int GAIN = NPARAM - 1;
constexpr int WCHUNK = 4096;           // rows per partial weight and bias gradient
constexpr int LOSS_BLK = 64;           // workgroups per sample in the loss

// training steps whose losses stay on the device: at most 1024, 16 MB of partial sums
int loss_steps(int max_batch) { return std::max(1, std::min(1024, (1 << 22) / LOSS_BLK / max_batch)); }

thread_local std::string g_cnn_err;

}  // namespace

struct plsqr_cnn {
    int nx = 0, ny = 0, nz = 0, V = 0, max_batch = 0;
    hipStream_t stream = nullptr;
    float *params = nullptr, *grads = nullptr, *adam_m = nullptr, *adam_v = nullptr;
    uint8_t *mask = nullptr;
    uint16_t *wf[LAYERS] = {}, *wb[LAYERS] = {};
    bool weights_dirty = true;
    uint16_t *act[LAYERS] = {};       // inputs of layers 1..3 (bf16, 32 channels; layer 0 reads xin)
    float *zout = nullptr, *dz1 = nullptr;  // output and its gradient, one channel
    uint16_t *dz[2] = {};             // gradients of the layers' outputs below
    float *wpart = nullptr, *bpart = nullptr, *lpart = nullptr;
    int *pick = nullptr;  // training pairs of loss_steps(max_batch) steps
    float *xin = nullptr, *tgt = nullptr, *tn = nullptr;
    int count = 0;
    float *data_in = nullptr, *data_t = nullptr, *data_tn = nullptr;
    size_t data_bytes = 0;
    long long adam_t = 0;
    float gain = 1.f;  // host copy of params[GAIN]
    std::vector<void *> allocs;
    size_t bytes = 0;
    std::string err;
};

namespace {

int set_err(plsqr_cnn *h, int code, const std::string &msg) {
    if (h) {
        if (h->err.empty()) h->err = msg;
    } else {
        g_cnn_err = msg;
    }
    return code;
}

#define CN_TRY(h, expr)                                                                       \
    do {                                                                                      \
        hipError_t e_ = (expr);                                                               \
        if (e_ != hipSuccess)                                                                 \
            return set_err(h, PLSQR_ERR_HIP, std::string(#expr) + ": " + hipGetErrorString(e_)); \
    } while (0)

#define CN_LAUNCH(h) CN_TRY(h, hipGetLastError())

template <class T>
int calloc_dev(plsqr_cnn *h, T **p, size_t count) {
    *p = nullptr;
    if (count == 0) count = 1;
    hipError_t e = hipMalloc((void **)p, sizeof(T) * count);
    if (e != hipSuccess) {
        *p = nullptr;
        return set_err(h, PLSQR_ERR_NOMEM,
                       "hipMalloc of " + std::to_string(sizeof(T) * count) + " bytes failed: " + hipGetErrorString(e));
    }
    h->allocs.push_back((void *)*p);
    h->bytes += sizeof(T) * count;
    return PLSQR_OK;
}

// Buffers of one call out of few allocations.  An hipMalloc and hipFree pair
// takes 4 us below 2 MiB and 16 to 27 from there, so up to 4 MiB are spread over
// allocations below it and more share one (in us, one per buffer / one in all /
// this rule: forward of 8192 voxels 192 / 218 / 169, of 11968 279 / 258 / 209;
// backward of 4096 398 / 267 / 225, of 9984, 5.9 MiB, 574 / 401 / 401, spread
// 428).  Each buffer starts on a 256-byte line.
struct CallBuffers {
    static constexpr size_t SMALL = (size_t)2 << 20;
    struct Part {
        void **p;
        size_t bytes;
    };
    std::vector<Part> parts;
    std::vector<void *> blocks;
    template <class T>
    void add(T **p, size_t count) {
        parts.push_back({(void **)p, (std::max<size_t>(sizeof(T) * count, 1) + 255) / 256 * 256});
    }
    int alloc(std::string &err) {
        size_t total = 0;
        for (const Part &q : parts) total += q.bytes;
        const size_t most = total <= 2 * SMALL ? SMALL : total + 1;  // an allocation stays below this
        for (size_t i = 0, j; i < parts.size(); i = j) {
            size_t bytes = 0;
            for (j = i; j < parts.size() && (j == i || bytes + parts[j].bytes < most); ++j) bytes += parts[j].bytes;
            void *block = nullptr;
            const hipError_t e = hipMalloc(&block, bytes);
            if (e != hipSuccess) {
                err = "hipMalloc of " + std::to_string(bytes) + " bytes failed: " + hipGetErrorString(e);
                return PLSQR_ERR_NOMEM;
            }
            blocks.push_back(block);
            char *at = (char *)block;
            for (size_t k = i; k < j; ++k) {
                *parts[k].p = at;
                at += parts[k].bytes;
            }
        }
        return PLSQR_OK;
    }
    ~CallBuffers() {
        for (void *b : blocks) (void)hipFree(b);
    }
};

void free_dev(plsqr_cnn *h, void *p) {
    auto it = std::find(h->allocs.begin(), h->allocs.end(), p);
    if (it != h->allocs.end()) {
        h->allocs.erase(it);
        (void)hipFree(p);
    }
}

int grid_for(long long work, int per, int cap) {
    long long g = (work + per - 1) / per;
    return (int)std::max(1LL, std::min<long long>(g, cap));
}

// SplitMix64 (Steele, Lea and Flood, 2014) and Box-Muller normals
struct Rng {
    uint64_t s;
    uint64_t next() {
        uint64_t z = (s += 0x9e3779b97f4a7c15ULL);
        z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ULL;
        z = (z ^ (z >> 27)) * 0x94d049bb133111ebULL;
        return z ^ (z >> 31);
    }
    double uniform() { return ((next() >> 11) + 0.5) * (1.0 / 9007199254740992.0); }
    double normal() {
        const double u1 = uniform(), u2 = uniform();
        return std::sqrt(-2.0 * std::log(u1)) * std::cos(6.283185307179586 * u2);
    }
};

// zero for the padded parameters: first layer input channels 1..31, last
// layer output channels 1..31 (weights and bias)
bool param_live(int i) {
    if (i == GAIN) return false;
    const int l = i / LSZ, j = i % LSZ;
    if (j < WSZ) {
        const int n = (j / C) % C, k = j % C;
        if (l == 0 && k != 0) return false;
        if (l == LAYERS - 1 && n != 0) return false;
        return true;
    }
    const int n = j - WSZ;
    return !(l == LAYERS - 1 && n != 0);
}

int prep_weights(plsqr_cnn *h) {
    if (!h->weights_dirty) return PLSQR_OK;
    for (int l = 0; l < LAYERS; ++l)
        hipLaunchKernelGGL(kc_prep_weights, dim3((WSZ + 255) / 256), dim3(256), 0, h->stream, h->params + (size_t)l * LSZ,
                           h->wf[l], h->wb[l]);
    CN_LAUNCH(h);
    h->weights_dirty = false;
    return PLSQR_OK;
}

// Compute units of the current device, looked up once per device.
int compute_units() {
    constexpr int MAX_DEVICES = 64;
    static std::atomic<int> known[MAX_DEVICES];
    int dev = 0, cu = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= MAX_DEVICES) return 256;
    if ((cu = known[dev].load(std::memory_order_relaxed)) > 0) return cu;
    if (hipDeviceGetAttribute(&cu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cu < 1) cu = 256;
    known[dev].store(cu, std::memory_order_relaxed);
    return cu;
}

// One convolution layer over `samples` grids.  By bricks (kc_conv): one workgroup
// per CU, or per brick where there are fewer; a multiple of eight when it can be,
// so that each XCD takes one range of bricks.  By rows (kc_conv_rows) where that
// takes fewer than half as many rounds over the CUs, a round being a brick or 256
// rows per CU: a round of bricks takes 3 to 8 us however few voxels they hold.
// FP32 layers in us, rounds and times by bricks against by rows: 131072 grids of
// one voxel 512 / 2, 1465 / 23; 1 x 1 x 131072 64 / 2, 262 / 23; 256 grids of
// 1 x 16 x 16 4 / 1, 31 / 14; 170 of 9^3 6 / 2, 51 / 22; 69 of 25 x 25 x 3 5 / 2,
// 31 / 26.  Below the line: 1024 of 5 x 4 x 4 4 / 2, 19.5 / 20.8; 512 of 3^3 2 / 1,
// 12.0 / 12.6; 200 x 2 x 200 3 / 2, 21 / 24; 32 of 16^3 1 / 2, 18 / 24.
template <int IN, bool WF32, int OUT>
void conv(int nx, int ny, int nz, int samples, const void *in, const void *w, const float *bias, const uint16_t *mask,
          int relu, void *out, hipStream_t st) {
    auto bricks = [](int n) { return (long long)((n + CB - 1) / CB); };
    const long long tiles = bricks(nx) * bricks(ny) * bricks(nz) * samples, rows = (long long)nx * ny * nz * samples;
    const int aligned = (((uintptr_t)in | (uintptr_t)out) & 15) == 0, cus = compute_units();
    const long long brick_rounds = (tiles + cus - 1) / cus, row_blocks = (rows + 32 * CB - 1) / (32 * CB);
    // the offsets within a brick's neighbourhood have 32 bits
    const bool wide = (long long)CH * nx * ny * 4 > UINT32_MAX;
    if (wide || brick_rounds > 2 * ((row_blocks + cus - 1) / cus)) {
        const long long g = std::min<long long>(row_blocks, cus);
        hipLaunchKernelGGL((kc_conv_rows<IN, WF32, OUT>), dim3((unsigned)g), dim3(CONV_THREADS), 0, st, nx, ny, nz, (unsigned)rows,
                           in, w, bias, mask, relu, out, aligned);
        return;
    }
    long long g = std::min<long long>(tiles, cus);
    if (g >= 8) g = g / 8 * 8;
    hipLaunchKernelGGL((kc_conv<IN, WF32, OUT>), dim3((unsigned)g), dim3(CONV_THREADS), 0, st, nx, ny, nz, samples, in, w,
                       bias, mask, relu, out, aligned);
}

// the network on h->xin (batch samples): activations act[0..3], zout
int forward(plsqr_cnn *h, int batch) {
    int rc;
    if ((rc = prep_weights(h))) return rc;
    for (int l = 0; l < LAYERS; ++l) {
        const float *bias = h->params + (size_t)l * LSZ + WSZ;
        const bool last = l == LAYERS - 1;
        if (l == 0)
            conv<CONV_ONE, false, CONV_BF16>(h->nx, h->ny, h->nz, batch, h->xin, h->wf[l], bias, nullptr, 1, h->act[1],
                                             h->stream);
        else if (!last)
            conv<CONV_BF16, false, CONV_BF16>(h->nx, h->ny, h->nz, batch, h->act[l], h->wf[l], bias, nullptr, 1,
                                              h->act[l + 1], h->stream);
        else
            conv<CONV_BF16, false, CONV_ONE>(h->nx, h->ny, h->nz, batch, h->act[l], h->wf[l], bias, nullptr, 0, h->zout,
                                             h->stream);
        CN_LAUNCH(h);
    }
    return PLSQR_OK;
}

// Weight and bias gradients of one layer; DONE: dout is one channel (FP32).  An
// error is left with h, or without a handle for plsqr_cnn_last_error(NULL).
template <bool DONE>
int wgrad(plsqr_cnn *h, int nx, int ny, int nz, long long total, const uint16_t *in, const void *dout, float *gw,
          float *gb, float *wpart, float *bpart, hipStream_t st) {
    const int nch = (int)((total + WCHUNK - 1) / WCHUNK);
    // nine taps per workgroup where a line fits and they fill the chip's 512
    // slots (two workgroups per CU), else three: three times as many workgroups
    // (a training step in us with nine / three: 67^3 x 4, 882 workgroups of nine,
    // 988 / 1027; 48^3 x 4, 324, 468 / 450; 67^3, 222, 388 / 374; 31 x 27 x 35 x 2,
    // 45, 284 / 236)
    const bool nine = nx <= WGRAD_NX9 && nch * 3 >= 512;
    const unsigned blocks = (unsigned)((nch * (nine ? 3 : 9) + 7) / 8 * 8);
    if (nine)
        hipLaunchKernelGGL((kc_wgrad<9, DONE>), dim3(blocks), dim3(256), 0, st, nx, ny, nz, total, WCHUNK, in, dout, wpart,
                           bpart);
    else
        hipLaunchKernelGGL((kc_wgrad<3, DONE>), dim3(blocks), dim3(256), 0, st, nx, ny, nz, total, WCHUNK, in, dout, wpart,
                           bpart);
    hipLaunchKernelGGL((kc_grad_reduce<false>), dim3(WSZ / GRAD_RED + 1), dim3(GRAD_RED), 0, st, nch, (const float *)wpart,
                       (const float *)bpart, gw, gb);
    return hipGetLastError() == hipSuccess ? PLSQR_OK : set_err(h, PLSQR_ERR_HIP, "gradient kernels failed to launch");
}

// The first layer's; its gradients of the padded input channels stay zero.
int wgrad_first(plsqr_cnn *h, long long total, const uint16_t *dout, float *gw, float *gb) {
    const int nch = (int)((total + WCHUNK - 1) / WCHUNK);
    hipLaunchKernelGGL(kc_wgrad_first, dim3(nch), dim3(256), 0, h->stream, h->nx, h->ny, h->nz, total, WCHUNK,
                       (const float *)h->xin, dout, h->wpart, h->bpart);
    hipLaunchKernelGGL((kc_grad_reduce<true>), dim3(C * C / GRAD_RED + 1), dim3(GRAD_RED), 0, h->stream, nch,
                       (const float *)h->wpart, (const float *)h->bpart, gw, gb);
    CN_LAUNCH(h);
    return PLSQR_OK;
}

// loss of zout against tgt/tn (batch samples) as partial sums in lpart, dz1 =
// its gradient
int loss_and_grad(plsqr_cnn *h, int batch, float *lpart) {
    hipLaunchKernelGGL(kc_loss, dim3(LOSS_BLK, batch), dim3(256), 0, h->stream, h->V, batch, LOSS_BLK,
                       (const float *)h->zout, (const float *)h->tgt, (const float *)h->tn, h->dz1, lpart);
    CN_LAUNCH(h);
    return PLSQR_OK;
}

// the loss from its partial sums and the samples' target norms
double loss_of(const float *part, const float *tn, int batch) {
    double L = 0.0;
    for (int s = 0; s < batch; ++s) {
        double e = 0.0;
        for (int b = 0; b < LOSS_BLK; ++b) e += part[(size_t)s * LOSS_BLK + b];
        L += e / tn[s];
    }
    return L / batch;
}

int backward(plsqr_cnn *h, int batch) {
    const long long total = (long long)batch * h->V;
    int cur = 0, rc;
    for (int l = LAYERS - 1; l >= 0; --l) {
        float *gw = h->grads + (size_t)l * LSZ;
        const bool last = l == LAYERS - 1;
        if (last)
            rc = wgrad<true>(h, h->nx, h->ny, h->nz, total, h->act[l], h->dz1, gw, gw + WSZ, h->wpart, h->bpart, h->stream);
        else if (l > 0)
            rc = wgrad<false>(h, h->nx, h->ny, h->nz, total, h->act[l], h->dz[cur], gw, gw + WSZ, h->wpart, h->bpart,
                              h->stream);
        else
            rc = wgrad_first(h, total, h->dz[cur], gw, gw + WSZ);
        if (rc) return rc;
        if (l == 0) break;
        // gradient of the layer's input, through the ReLU of layer l-1
        if (last) {
            conv<CONV_ONE, false, CONV_BF16>(h->nx, h->ny, h->nz, batch, h->dz1, h->wb[l], nullptr, h->act[l], 0, h->dz[cur],
                                             h->stream);
        } else {
            conv<CONV_BF16, false, CONV_BF16>(h->nx, h->ny, h->nz, batch, h->dz[cur], h->wb[l], nullptr, h->act[l], 0,
                                              h->dz[1 - cur], h->stream);
            cur = 1 - cur;
        }
        CN_LAUNCH(h);
    }
    return PLSQR_OK;
}

// normalised copies of caller samples: in = atb / s, t = x / s, s = rms(atb)
void normalise(int V, const double *atb, const double *xs, double gain, std::vector<float> &in, std::vector<float> &t,
               float *tn, double *scale) {
    double ss = 0.0;
    for (int v = 0; v < V; ++v) ss += atb[v] * atb[v];
    double s = std::sqrt(ss / V);
    if (!(s > 0.0) || !std::isfinite(s)) s = 1.0;
    *scale = s;
    double tt = 0.0;
    for (int v = 0; v < V; ++v) {
        in[(size_t)v] = (float)(atb[v] / s);
        if (xs) {
            const double q = xs[v] / s / gain;
            t[(size_t)v] = (float)q;
            tt += q * q;
        }
    }
    if (tn) *tn = (float)(tt > 0.0 ? tt : 1.0);
}

int check(plsqr_cnn *h) {
    if (!h) return PLSQR_ERR_ARG;
    if (h->allocs.empty()) return set_err(h, PLSQR_ERR_STATE, "network failed to initialise");
    return PLSQR_OK;
}

// load `batch` caller samples into xin/tgt/tn
int load_samples(plsqr_cnn *h, int batch, const double *atb, const double *xs, std::vector<double> *scales) {
    std::vector<float> in((size_t)h->V), t((size_t)h->V);
    std::vector<float> tn((size_t)batch, 1.f);
    if (scales) scales->assign((size_t)batch, 1.0);
    for (int s = 0; s < batch; ++s) {
        double sc;
        normalise(h->V, atb + (size_t)s * h->V, xs ? xs + (size_t)s * h->V : nullptr, h->gain, in, t, &tn[(size_t)s],
                  &sc);
        if (scales) (*scales)[(size_t)s] = sc;
        CN_TRY(h, hipMemcpyAsync(h->xin + (size_t)s * h->V, in.data(), sizeof(float) * h->V, hipMemcpyHostToDevice,
                                 h->stream));
        if (xs)
            CN_TRY(h, hipMemcpyAsync(h->tgt + (size_t)s * h->V, t.data(), sizeof(float) * h->V, hipMemcpyHostToDevice,
                                     h->stream));
        CN_TRY(h, hipStreamSynchronize(h->stream));  // the host vectors are reused
    }
    CN_TRY(h, hipMemcpyAsync(h->tn, tn.data(), sizeof(float) * batch, hipMemcpyHostToDevice, h->stream));
    CN_TRY(h, hipStreamSynchronize(h->stream));
    return PLSQR_OK;
}

}  // namespace

// ---------------------------------------------------------------------------
// Allocation-free variant of plsqr_cnn_conv_forward for callers that cannot
// allocate device memory (HIP graph capture, serving loops): the layer kernels
// round the FP32 operands themselves.  A call whose output overlaps its input or weights
// needs copies of them first; that scratch -- the bf16 input and weights -- lives
// in one file-scope device array, fixed in size; each device holds its own copy,
// found once per device with hipGetSymbolAddress.  Every element the kernels read
// is written earlier in the same call, so no clearing is needed; such calls that
// overlap on one device share the array and race.
// ---------------------------------------------------------------------------
constexpr long long NOALLOC_MAX_ELEMS = 1LL << 22;  // batch * voxels * 32 channels of input
constexpr size_t NOALLOC_BYTES = sizeof(uint16_t) * ((size_t)NOALLOC_MAX_ELEMS + (size_t)WSZ);
static __device__ __align__(256) unsigned char scratch[NOALLOC_BYTES];

namespace {
constexpr int MAX_DEVICES = 64;
std::mutex g_scratch_mu;
void *g_scratch_ptr[MAX_DEVICES] = {};

// The current device's address of `scratch` (looked up on the first call on
// that device, with that device current).
int scratch_ptr(void **out) {
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return set_err(nullptr, PLSQR_ERR_HIP, std::string("hipGetDevice: ") + hipGetErrorString(e));
    if (dev < 0 || dev >= MAX_DEVICES) return set_err(nullptr, PLSQR_ERR_STATE, "device ordinal out of range");
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void *p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p)
            return set_err(nullptr, PLSQR_ERR_HIP, std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
        g_scratch_ptr[dev] = p;
    }
    *out = g_scratch_ptr[dev];
    return PLSQR_OK;
}

bool overlap(const void *a, size_t na, const void *b, size_t nb) {
    const uintptr_t x = (uintptr_t)a, y = (uintptr_t)b;
    return x < y + nb && y < x + na;
}
}  // namespace

extern "C" {

const char *plsqr_cnn_last_error(const plsqr_cnn *h) { return h ? h->err.c_str() : g_cnn_err.c_str(); }

int plsqr_cnn_param_count(void) { return NPARAM; }

void plsqr_cnn_destroy(plsqr_cnn *h) {
    if (!h) return;
    if (h->stream) (void)hipStreamSynchronize(h->stream);
    for (void *p : h->allocs) (void)hipFree(p);
    if (h->stream) (void)hipStreamDestroy(h->stream);
    delete h;
}

int plsqr_cnn_create(int nx, int ny, int nz, int max_batch, unsigned long long seed, plsqr_cnn **out) {
    g_cnn_err.clear();
    if (!out) return PLSQR_ERR_ARG;
    *out = nullptr;
    if (nx < 1 || ny < 1 || nz < 1 || max_batch < 1 || (long long)nx * ny * nz > (1LL << 26) ||
        (long long)nx * ny * nz * max_batch * C > (1LL << 33))
        return set_err(nullptr, PLSQR_ERR_ARG, "grid or batch out of range");
    plsqr_cnn *h = new plsqr_cnn();
    h->nx = nx;
    h->ny = ny;
    h->nz = nz;
    h->V = nx * ny * nz;
    h->max_batch = max_batch;
    auto fail = [&](int code) {
        g_cnn_err = h->err;
        plsqr_cnn_destroy(h);
        return code;
    };
    hipError_t e = hipStreamCreateWithFlags(&h->stream, hipStreamNonBlocking);
    if (e != hipSuccess) return fail(set_err(h, PLSQR_ERR_HIP, std::string("hipStreamCreate: ") + hipGetErrorString(e)));
    const long long total = (long long)max_batch * h->V;
    const int nch = (int)((total + WCHUNK - 1) / WCHUNK);
    int rc;
    if ((rc = calloc_dev(h, &h->params, NPARAM)) || (rc = calloc_dev(h, &h->grads, NPARAM)) ||
        (rc = calloc_dev(h, &h->adam_m, NPARAM)) || (rc = calloc_dev(h, &h->adam_v, NPARAM)) ||
        (rc = calloc_dev(h, &h->mask, NPARAM)) || (rc = calloc_dev(h, &h->zout, (size_t)total)) ||
        (rc = calloc_dev(h, &h->dz1, (size_t)total)) ||
        (rc = calloc_dev(h, &h->dz[0], (size_t)total * C)) || (rc = calloc_dev(h, &h->dz[1], (size_t)total * C)) ||
        (rc = calloc_dev(h, &h->wpart, (size_t)nch * TAPS * C * C)) || (rc = calloc_dev(h, &h->bpart, (size_t)nch * C)) ||
        (rc = calloc_dev(h, &h->lpart, (size_t)loss_steps(max_batch) * max_batch * LOSS_BLK)) ||
        (rc = calloc_dev(h, &h->pick, (size_t)loss_steps(max_batch) * max_batch)) || (rc = calloc_dev(h, &h->xin, (size_t)total)) ||
        (rc = calloc_dev(h, &h->tgt, (size_t)total)) || (rc = calloc_dev(h, &h->tn, (size_t)max_batch)))
        return fail(rc);
    for (int l = 0; l < LAYERS; ++l)
        if ((rc = calloc_dev(h, &h->wf[l], WSZ)) || (rc = calloc_dev(h, &h->wb[l], WSZ)) ||
            (l > 0 && (rc = calloc_dev(h, &h->act[l], (size_t)total * C))))
            return fail(rc);
    // He initialisation (fan-in = 27 x real input channels), zero biases
    std::vector<float> p((size_t)NPARAM, 0.f);
    std::vector<uint8_t> m((size_t)NPARAM, 0);
    Rng rng{seed};
    for (int i = 0; i < NPARAM; ++i) {
        m[(size_t)i] = param_live(i) ? 1 : 0;
        const int l = i / LSZ, j = i % LSZ;
        if (!m[(size_t)i] || j >= WSZ) continue;
        const double fan_in = TAPS * (l == 0 ? 1.0 : (double)C);
        const double sd = std::sqrt((l == LAYERS - 1 ? 1.0 : 2.0) / fan_in);
        p[(size_t)i] = (float)(sd * rng.normal());
    }
    p[GAIN] = 1.f;
    e = hipMemcpy(h->params, p.data(), sizeof(float) * NPARAM, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(h->mask, m.data(), NPARAM, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemset(h->adam_m, 0, sizeof(float) * NPARAM);
    if (e == hipSuccess) e = hipMemset(h->adam_v, 0, sizeof(float) * NPARAM);
    if (e == hipSuccess) e = hipMemset(h->grads, 0, sizeof(float) * NPARAM);
    if (e != hipSuccess) return fail(set_err(h, PLSQR_ERR_HIP, std::string("initialise: ") + hipGetErrorString(e)));
    *out = h;
    return PLSQR_OK;
}

size_t plsqr_cnn_device_bytes(const plsqr_cnn *h) { return h ? h->bytes : 0; }

int plsqr_cnn_get_params(plsqr_cnn *h, float *params) {
    int rc;
    if ((rc = check(h))) return rc;
    if (!params) return set_err(h, PLSQR_ERR_ARG, "params is NULL");
    CN_TRY(h, hipMemcpyAsync(params, h->params, sizeof(float) * NPARAM, hipMemcpyDeviceToHost, h->stream));
    CN_TRY(h, hipStreamSynchronize(h->stream));
    return PLSQR_OK;
}

int plsqr_cnn_set_params(plsqr_cnn *h, const float *params) {
    int rc;
    if ((rc = check(h))) return rc;
    if (!params) return set_err(h, PLSQR_ERR_ARG, "params is NULL");
    for (int i = 0; i < NPARAM; ++i) {
        if (!std::isfinite(params[i])) return set_err(h, PLSQR_ERR_NONFINITE, "parameter " + std::to_string(i) + " is not finite");
        if (i != GAIN && !param_live(i) && params[i] != 0.f)
            return set_err(h, PLSQR_ERR_ARG, "parameter " + std::to_string(i) + " is a padded entry and must be 0");
    }
    if (!(params[GAIN] > 0.f)) return set_err(h, PLSQR_ERR_ARG, "the output gain must be positive");
    h->gain = params[GAIN];
    CN_TRY(h, hipMemcpyAsync(h->params, params, sizeof(float) * NPARAM, hipMemcpyHostToDevice, h->stream));
    CN_TRY(h, hipStreamSynchronize(h->stream));
    h->weights_dirty = true;
    return PLSQR_OK;
}

int plsqr_cnn_set_data(plsqr_cnn *h, int count, const double *atb, const double *xstar) {
    int rc;
    if ((rc = check(h))) return rc;
    if (count < 1 || !atb || !xstar) return set_err(h, PLSQR_ERR_ARG, "count, atb and xstar are required");
    for (float **p : {&h->data_in, &h->data_t, &h->data_tn})
        if (*p) {
            free_dev(h, *p);
            *p = nullptr;
        }
    h->count = 0;
    if ((rc = calloc_dev(h, &h->data_in, (size_t)count * h->V)) || (rc = calloc_dev(h, &h->data_t, (size_t)count * h->V)) ||
        (rc = calloc_dev(h, &h->data_tn, (size_t)count)))
        return rc;
    std::vector<float> in((size_t)h->V), t((size_t)h->V), tn((size_t)count);
    // output gain: the RMS of the scaled targets x*/s over the set, so that
    // the network's output channel is of order one
    double gsum = 0.0;
    for (int s = 0; s < count; ++s) {
        const double *a = atb + (size_t)s * h->V, *x = xstar + (size_t)s * h->V;
        double aa = 0.0, xx = 0.0;
        for (int v = 0; v < h->V; ++v) {
            if (!std::isfinite(a[v]) || !std::isfinite(x[v]))
                return set_err(h, PLSQR_ERR_NONFINITE, "sample " + std::to_string(s) + " holds a NaN or Inf");
            aa += a[v] * a[v];
            xx += x[v] * x[v];
        }
        if (aa > 0.0) gsum += xx / aa;  // mean((x/s)^2) with s^2 = aa / V
    }
    const double g = std::sqrt(gsum / count);
    h->gain = (float)(g > 0.0 && std::isfinite(g) ? g : 1.0);
    CN_TRY(h, hipMemcpyAsync(h->params + GAIN, &h->gain, sizeof(float), hipMemcpyHostToDevice, h->stream));
    for (int s = 0; s < count; ++s) {
        double sc;
        const double *a = atb + (size_t)s * h->V, *x = xstar + (size_t)s * h->V;
        normalise(h->V, a, x, h->gain, in, t, &tn[(size_t)s], &sc);
        CN_TRY(h, hipMemcpyAsync(h->data_in + (size_t)s * h->V, in.data(), sizeof(float) * h->V, hipMemcpyHostToDevice,
                                 h->stream));
        CN_TRY(h, hipMemcpyAsync(h->data_t + (size_t)s * h->V, t.data(), sizeof(float) * h->V, hipMemcpyHostToDevice,
                                 h->stream));
        CN_TRY(h, hipStreamSynchronize(h->stream));
    }
    CN_TRY(h, hipMemcpyAsync(h->data_tn, tn.data(), sizeof(float) * count, hipMemcpyHostToDevice, h->stream));
    CN_TRY(h, hipStreamSynchronize(h->stream));
    h->count = count;
    return PLSQR_OK;
}

int plsqr_cnn_train(plsqr_cnn *h, int steps, int batch, float lr, unsigned long long seed, double *loss_out) {
    int rc;
    if ((rc = check(h))) return rc;
    if (h->count < 1) return set_err(h, PLSQR_ERR_STATE, "no training data (plsqr_cnn_set_data)");
    if (batch < 1 || batch > h->max_batch || batch > h->count || steps < 0 || !(lr > 0.f))
        return set_err(h, PLSQR_ERR_ARG, "bad steps, batch or learning rate");
    std::vector<int> order((size_t)h->count);
    Rng rng{seed};
    size_t pos = order.size();
    const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
    LayerWeights lw;
    static_assert(LAYERS <= MAX_LAYERS, "a pair of weight arrays per layer");
    for (int l = 0; l < LAYERS; ++l) {
        lw.wf[l] = h->wf[l];
        lw.wb[l] = h->wb[l];
    }
    std::vector<int> pick;
    std::vector<float> part, tn((size_t)h->count);
    CN_TRY(h, hipMemcpyAsync(tn.data(), h->data_tn, sizeof(float) * tn.size(), hipMemcpyDeviceToHost, h->stream));
    CN_TRY(h, hipStreamSynchronize(h->stream));
    // the picks of many steps go to the device together and their losses come
    // back together, so the steps are queued without waiting
    const int group = loss_steps(h->max_batch);
    for (int it0 = 0; it0 < steps; it0 += group) {
        const int n = std::min(group, steps - it0);
        pick.resize((size_t)n * batch);
        for (int &p : pick) {
            if (pos >= order.size()) {  // a new epoch: Fisher-Yates shuffle
                for (int i = 0; i < h->count; ++i) order[(size_t)i] = i;
                for (int i = h->count - 1; i > 0; --i) std::swap(order[(size_t)i], order[(size_t)(rng.next() % (uint64_t)(i + 1))]);
                pos = 0;
            }
            p = order[pos++];
        }
        CN_TRY(h, hipMemcpyAsync(h->pick, pick.data(), sizeof(int) * pick.size(), hipMemcpyHostToDevice, h->stream));
        for (int it = 0; it < n; ++it) {
            // a copy: blocks enough for every CU (67^3 x 4: 64 per sample 13.3 us, 512 6.3)
            hipLaunchKernelGGL(kc_pick, dim3(grid_for(h->V, 256, 512), batch), dim3(256), 0, h->stream, h->V, batch, it,
                               (const int *)h->pick, (const float *)h->data_in, (const float *)h->data_t,
                               (const float *)h->data_tn, h->xin, h->tgt, h->tn);
            CN_LAUNCH(h);
            if ((rc = forward(h, batch)) || (rc = loss_and_grad(h, batch, h->lpart + (size_t)it * batch * LOSS_BLK)) ||
                (rc = backward(h, batch)))
                return rc;
            ++h->adam_t;
            const float c1 = 1.f - std::pow(b1, (float)h->adam_t), c2 = 1.f - std::pow(b2, (float)h->adam_t);
            hipLaunchKernelGGL(kc_adam, dim3((NPARAM + 255) / 256), dim3(256), 0, h->stream, NPARAM, h->params,
                               (const float *)h->grads, h->adam_m, h->adam_v, (const uint8_t *)h->mask, lr, b1, b2, eps, c1,
                               c2, LSZ, lw);
            CN_LAUNCH(h);
        }
        part.resize((size_t)n * batch * LOSS_BLK);
        CN_TRY(h, hipMemcpyAsync(part.data(), h->lpart, sizeof(float) * part.size(), hipMemcpyDeviceToHost, h->stream));
        CN_TRY(h, hipStreamSynchronize(h->stream));
        std::vector<float> tb((size_t)batch);
        for (int it = 0; loss_out && it < n; ++it) {
            for (int s = 0; s < batch; ++s) tb[(size_t)s] = tn[(size_t)pick[(size_t)it * batch + s]];
            loss_out[it0 + it] = loss_of(part.data() + (size_t)it * batch * LOSS_BLK, tb.data(), batch);
        }
    }
    return PLSQR_OK;
}

int plsqr_cnn_gradient(plsqr_cnn *h, int batch, const double *atb, const double *xstar, float *grads, double *loss) {
    int rc;
    if ((rc = check(h))) return rc;
    if (batch < 1 || batch > h->max_batch || !atb || !xstar || !grads || !loss)
        return set_err(h, PLSQR_ERR_ARG, "bad gradient arguments");
    if ((rc = load_samples(h, batch, atb, xstar, nullptr))) return rc;
    if ((rc = forward(h, batch)) || (rc = loss_and_grad(h, batch, h->lpart)) || (rc = backward(h, batch))) return rc;
    std::vector<float> part((size_t)batch * LOSS_BLK), tn((size_t)batch);
    CN_TRY(h, hipMemcpyAsync(part.data(), h->lpart, sizeof(float) * part.size(), hipMemcpyDeviceToHost, h->stream));
    CN_TRY(h, hipMemcpyAsync(tn.data(), h->tn, sizeof(float) * tn.size(), hipMemcpyDeviceToHost, h->stream));
    CN_TRY(h, hipMemcpyAsync(grads, h->grads, sizeof(float) * NPARAM, hipMemcpyDeviceToHost, h->stream));
    CN_TRY(h, hipStreamSynchronize(h->stream));
    *loss = loss_of(part.data(), tn.data(), batch);
    return PLSQR_OK;
}

int plsqr_cnn_predict(plsqr_cnn *h, int count, const double *atb, double *x0) {
    int rc;
    if ((rc = check(h))) return rc;
    if (count < 0 || (count > 0 && (!atb || !x0))) return set_err(h, PLSQR_ERR_ARG, "atb and x0 are required");
    std::vector<float> z((size_t)h->V);
    for (int s0 = 0; s0 < count; s0 += h->max_batch) {
        const int nb = std::min(h->max_batch, count - s0);
        std::vector<double> scales;
        if ((rc = load_samples(h, nb, atb + (size_t)s0 * h->V, nullptr, &scales)) || (rc = forward(h, nb))) return rc;
        for (int s = 0; s < nb; ++s) {
            CN_TRY(h, hipMemcpyAsync(z.data(), h->zout + (size_t)s * h->V, sizeof(float) * z.size(),
                                     hipMemcpyDeviceToHost, h->stream));
            CN_TRY(h, hipStreamSynchronize(h->stream));
            double *o = x0 + (size_t)(s0 + s) * h->V;
            const double f = scales[(size_t)s] * (double)h->gain;
            for (int v = 0; v < h->V; ++v) o[v] = f * (double)z[(size_t)v];
        }
    }
    return PLSQR_OK;
}

// One 32 -> 32 convolution layer through the MFMA kernels, host arrays
// (operands rounded to bf16 inside; results in FP32).
int plsqr_cnn_conv_forward(int nx, int ny, int nz, int batch, const float *in, const float *w, const float *bias,
                           int relu, float *out) {
    g_cnn_err.clear();
    if (nx < 1 || ny < 1 || nz < 1 || batch < 1 || !in || !w || !out) return set_err(nullptr, PLSQR_ERR_ARG, "bad arguments");
    const long long total = (long long)batch * nx * ny * nz;
    float *din = nullptr, *dw = nullptr, *db = nullptr, *dout = nullptr;
    CallBuffers mem;
    mem.add(&din, (size_t)total * C);
    mem.add(&dw, WSZ);
    mem.add(&db, C);
    mem.add(&dout, (size_t)total * C);
    if (int rc = mem.alloc(g_cnn_err)) return rc;
    hipError_t e = hipMemcpy(din, in, sizeof(float) * total * C, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(dw, w, sizeof(float) * WSZ, hipMemcpyHostToDevice);
    if (e == hipSuccess && bias) e = hipMemcpy(db, bias, sizeof(float) * C, hipMemcpyHostToDevice);
    if (e == hipSuccess) {
        conv<CONV_F32, true, CONV_F32>(nx, ny, nz, batch, din, dw, bias ? db : nullptr, nullptr, relu, dout, 0);
        e = hipGetLastError();
        if (e == hipSuccess) e = hipDeviceSynchronize();
        if (e == hipSuccess) e = hipMemcpy(out, dout, sizeof(float) * total * C, hipMemcpyDeviceToHost);
    }
    if (e != hipSuccess) return set_err(nullptr, PLSQR_ERR_HIP, std::string("conv forward: ") + hipGetErrorString(e));
    return PLSQR_OK;
}

// plsqr_cnn_conv_forward on device pointers with the scratch above: no allocation.
int plsqr_cnn_conv_forward_noalloc(int nx, int ny, int nz, int batch, const float *in_dev, const float *w_dev,
                                   const float *bias_dev, int relu, float *out_dev, void *stream) {
    g_cnn_err.clear();
    if (nx < 1 || ny < 1 || nz < 1 || batch < 1 || !in_dev || !w_dev || !out_dev)
        return set_err(nullptr, PLSQR_ERR_ARG, "bad arguments");
    const long long total = (long long)batch * nx * ny * nz;
    if (total > NOALLOC_MAX_ELEMS / C)
        return set_err(nullptr, PLSQR_ERR_ARG,
                       "batch * nx * ny * nz = " + std::to_string(total) + " exceeds the allocation-free limit of " +
                           std::to_string(NOALLOC_MAX_ELEMS / C) + " voxels");
    const hipStream_t st = (hipStream_t)stream;
    const size_t out_bytes = sizeof(float) * (size_t)total * C;
    if (!overlap(in_dev, out_bytes, out_dev, out_bytes) && !overlap(w_dev, sizeof(float) * WSZ, out_dev, out_bytes)) {
        conv<CONV_F32, true, CONV_F32>(nx, ny, nz, batch, in_dev, w_dev, bias_dev, nullptr, relu, out_dev, st);
    } else {  // in place: the operands are copied to the scratch first
        void *base = nullptr;
        int rc = scratch_ptr(&base);
        if (rc) return rc;
        uint16_t *bin = (uint16_t *)base;
        uint16_t *wf = bin + NOALLOC_MAX_ELEMS;
        hipLaunchKernelGGL(kc_to_bf16, dim3(grid_for(total * C, 256, 4096)), dim3(256), 0, st, total * C, in_dev, bin);
        hipLaunchKernelGGL(kc_prep_weights, dim3((WSZ + 255) / 256), dim3(256), 0, st, w_dev, wf, (uint16_t *)nullptr);
        conv<CONV_BF16, false, CONV_F32>(nx, ny, nz, batch, bin, wf, bias_dev, nullptr, relu, out_dev, st);
    }
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return set_err(nullptr, PLSQR_ERR_HIP, std::string("conv forward: ") + hipGetErrorString(e));
    return PLSQR_OK;
}

// Gradients of one layer: din = data gradient (no ReLU mask), dw, dbias.
int plsqr_cnn_conv_backward(int nx, int ny, int nz, int batch, const float *in, const float *w, const float *dout,
                            float *din, float *dw, float *dbias) {
    g_cnn_err.clear();
    if (nx < 1 || ny < 1 || nz < 1 || batch < 1 || !in || !w || !dout || !din || !dw || !dbias)
        return set_err(nullptr, PLSQR_ERR_ARG, "bad arguments");
    const long long total = (long long)batch * nx * ny * nz;
    const int nch = (int)((total + WCHUNK - 1) / WCHUNK);
    float *fin = nullptr, *fw = nullptr, *fdo = nullptr, *fdi = nullptr, *gw = nullptr, *wpart = nullptr, *bpart = nullptr;
    uint16_t *bin = nullptr, *bdo = nullptr, *wb = nullptr;
    CallBuffers mem;
    mem.add(&fin, (size_t)total * C);
    mem.add(&fw, WSZ);
    mem.add(&fdo, (size_t)total * C);
    mem.add(&fdi, (size_t)total * C);
    mem.add(&gw, LSZ);
    mem.add(&wpart, (size_t)nch * TAPS * C * C);
    mem.add(&bpart, (size_t)nch * C);
    mem.add(&bin, (size_t)total * C);
    mem.add(&bdo, (size_t)total * C);
    mem.add(&wb, WSZ);
    int rc;
    if ((rc = mem.alloc(g_cnn_err))) return rc;
    hipError_t e = hipMemcpy(fin, in, sizeof(float) * total * C, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(fw, w, sizeof(float) * WSZ, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(fdo, dout, sizeof(float) * total * C, hipMemcpyHostToDevice);
    if (e == hipSuccess) {
        const int g = grid_for(total * C, 256, 4096);
        hipLaunchKernelGGL(kc_to_bf16, dim3(g), dim3(256), 0, 0, total * C, (const float *)fin, bin);
        hipLaunchKernelGGL(kc_to_bf16, dim3(g), dim3(256), 0, 0, total * C, (const float *)fdo, bdo);
        hipLaunchKernelGGL(kc_prep_weights, dim3((WSZ + 255) / 256), dim3(256), 0, 0, (const float *)fw, (uint16_t *)nullptr, wb);
        conv<CONV_BF16, false, CONV_F32>(nx, ny, nz, batch, bdo, wb, nullptr, nullptr, 0, fdi, 0);
        rc = wgrad<false>(nullptr, nx, ny, nz, total, bin, bdo, gw, gw + WSZ, wpart, bpart, 0);
        e = hipGetLastError();
        if (e == hipSuccess) e = hipDeviceSynchronize();
        if (e == hipSuccess) e = hipMemcpy(din, fdi, sizeof(float) * total * C, hipMemcpyDeviceToHost);
        if (e == hipSuccess) e = hipMemcpy(dw, gw, sizeof(float) * WSZ, hipMemcpyDeviceToHost);
        if (e == hipSuccess) e = hipMemcpy(dbias, gw + WSZ, sizeof(float) * C, hipMemcpyDeviceToHost);
    }
    if (e != hipSuccess) return set_err(nullptr, PLSQR_ERR_HIP, std::string("conv backward: ") + hipGetErrorString(e));
    return rc;
}

}  // extern "C"
