// gradhip engine: device model, paged KV cache, the per-token step (eager,
// hipGraph-replayed), the on-GPU generate loop, and the C ABI of
// include/gradhip.h.
#include "../../include/gradhip.h"
#include "checkpoint.h"
#include "tokenizer.h"
#include "kernels_attn.h"
#include "kernel_tables.h"
#include "kernels_common.h"
#include "kernels_gemm.h"
#include "kernels_gemv.h"
#include "kernels_pick.h"
#include "rows.h"

#include <algorithm>
#include <atomic>
#include <climits>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <exception>
#include <memory>
#include <mutex>
#include <numeric>
#include <string>
#include <tuple>
#include <vector>

namespace gh {

// ------------------------------------------------------------------ errors

struct ApiError {
    gh_status code;
    std::string msg;
};

static thread_local std::string g_last_error;

[[noreturn]] static void throw_device(hipError_t e, const char* what, const char* file, int line) {
    throw ApiError{GH_ERR_DEVICE, std::string("HIP error in ") + what + ": " + hipGetErrorString(e)
                                      + " (" + file + ":" + std::to_string(line) + ")"};
}

#define HIP_CHECK(expr)                                                        \
    do {                                                                       \
        hipError_t e_ = (expr);                                                \
        if (e_ != hipSuccess) throw_device(e_, #expr, __FILE__, __LINE__);     \
    } while (0)

template <typename F>
static gh_status guard(F&& f) {
    try {
        f();
        return GH_OK;
    } catch (const ApiError& e) {
        g_last_error = e.msg;
        return e.code;
    } catch (const std::out_of_range& e) {
        g_last_error = e.what();
        return GH_ERR_OUT_OF_RANGE;
    } catch (const std::invalid_argument& e) {
        g_last_error = e.what();
        return GH_ERR_INVALID_ARGUMENT;
    } catch (const std::bad_alloc&) {
        g_last_error = "out of host memory";
        return GH_ERR_RUNTIME;
    } catch (const std::exception& e) {
        g_last_error = e.what();
        return GH_ERR_RUNTIME;
    }
}

static void require_gpu() {
    int n = 0;
    hipError_t e = hipGetDeviceCount(&n);
    if (e != hipSuccess || n <= 0) {
        throw ApiError{GH_ERR_DEVICE,
                       "gradhip needs a gfx950 GPU: no HIP device is usable and there is no CPU "
                       "fallback"};
    }
}

// Device memory that a call is faster with and can do without, uncleared: false, and nothing
// allocated, if there is not enough.
template <typename T>
static bool try_alloc(T*& p, size_t n) {
    p = nullptr;
    const size_t bytes = std::max<size_t>(n, 1) * sizeof(T);
    // Test aid: no allocation of this kind above so many bytes.
    if (const char* most = std::getenv("GRADHIP_TEST_SPARE_BYTES"))
        if (bytes > std::strtoull(most, nullptr, 10)) return false;
    const hipError_t e = hipMalloc(&p, bytes);
    if (e == hipErrorOutOfMemory) {
        (void)hipGetLastError();  // (a later launch's check would find it)
        p = nullptr;
        return false;
    }
    HIP_CHECK(e);
    return true;
}

// ------------------------------------------------------------ device model

// Layout kernels.  Matrices arrive (in, out) row-major as grad.cpp stores them
// (inference.cpp:13) and are kept (out, in) so that one output's weights are a
// contiguous stream.  dst row of source column c is c * row_mul + row_off.
__global__ void transpose_in_kernel(const float* __restrict__ src, int rows, int cols,
                                    float* __restrict__ dst, int row_mul, int row_off) {
    __shared__ float tile[32][33];
    const int c0 = blockIdx.x * 32, r0 = blockIdx.y * 32;
    for (int i = threadIdx.y; i < 32; i += blockDim.y) {
        const int r = r0 + i, c = c0 + threadIdx.x;
        if (r < rows && c < cols) tile[i][threadIdx.x] = src[static_cast<size_t>(r) * cols + c];
    }
    __syncthreads();
    for (int i = threadIdx.y; i < 32; i += blockDim.y) {
        const int c = c0 + i, r = r0 + threadIdx.x;
        if (r < rows && c < cols)
            dst[(static_cast<size_t>(c) * row_mul + row_off) * rows + r] = tile[threadIdx.x][i];
    }
}

__global__ void transpose_out_kernel(const float* __restrict__ dev, int rows, int cols,
                                     float* __restrict__ out, int row_mul, int row_off) {
    __shared__ float tile[32][33];
    const int c0 = blockIdx.x * 32, r0 = blockIdx.y * 32;
    for (int i = threadIdx.y; i < 32; i += blockDim.y) {
        const int c = c0 + i, r = r0 + threadIdx.x;
        if (r < rows && c < cols)
            tile[threadIdx.x][i] = dev[(static_cast<size_t>(c) * row_mul + row_off) * rows + r];
    }
    __syncthreads();
    for (int i = threadIdx.y; i < 32; i += blockDim.y) {
        const int r = r0 + i, c = c0 + threadIdx.x;
        if (r < rows && c < cols) out[static_cast<size_t>(r) * cols + c] = tile[i][threadIdx.x];
    }
}

struct LayerWeights {
    float *wqkv, *bqkv;  // (3d, d), 3d
    float *wo, *bo;      // (d, d), d
    float *w1, *b1;      // GPT-2: (F, d), F.  Modern: (2F, d) rows (gate_p, up_p) interleaved
    float *w2, *b2;      // (d, F), d (GPT-2 only)
    float *g1, *be1, *g2, *be2;
};

// The split forms of a layer's matrices, for passes over many rows (kernels_split.h).
struct SplitLayer {
    char *wqkv, *wo, *w1, *w2;
};

// The same matrices in pairs (kernels_pair.h), each with its outputs' units, and the powers of two that the
// operands of those products are scaled by: norm(x) in front of QKV, keys, values and the attention's rows, norm(x) in front
// of FFN1, the hidden units.
struct PairLayer {
    char *wqkv, *wo, *w1, *w2;
    float *uqkv, *uo, *u1, *u2;
    int norm1, keys, attn, norm2, hidden;
};

// Device memory that is given back, also where making what it is for throws.
struct DeviceBlob {
    char* at = nullptr;
    DeviceBlob() = default;
    DeviceBlob(const DeviceBlob&) = delete;
    DeviceBlob& operator=(const DeviceBlob&) = delete;
    ~DeviceBlob() {
        if (at) (void)hipFree(at);
    }
};

// Split matrices in one allocation: there is one once they are ready.
struct SplitForm {
    std::mutex mutex;
    DeviceBlob blob;
    bool ready = false;
    bool unfit = false;  // the weights have no such form
};

// Where tensor i of the file lives on the device.
struct Placement {
    float* dst;
    bool transpose;
    int row_mul, row_off;
};

struct Model {
    Shape shape;
    std::optional<Fingerprint> tokenizer;
    float* blob = nullptr;
    size_t blob_floats = 0;
    float* E = nullptr;
    float* P = nullptr;
    std::vector<LayerWeights> layers;
    float *gf = nullptr, *bf = nullptr;
    float *rope_cos = nullptr, *rope_sin = nullptr;  // (max_len, head_size/2)
    std::vector<Placement> place;                    // file order

    // Split forms of the matrices, each written by the first pass that multiplies by it and kept: in pairs (four bytes
    // per weight beside the four above) or in three parts (six); the layers', and that of the logits matrix, which
    // scoring alone needs and at any length.
    mutable SplitForm layers_split, layers_pairs, logits_split, logits_pairs;
    mutable std::vector<SplitLayer> split_layers;
    mutable std::vector<PairLayer> pair_layers;
    mutable float* logits_unit = nullptr;  // of the logits matrix in pairs, in its allocation
    mutable int logits_norm = 0;             // the power of two of its operand, norm(x)

    // The XCD-sharded persistent kernel reads the weights from a second copy laid
    // out as one contiguous stream per workgroup (kernels_xcd.h); built by the
    // first session that uses it.
    mutable std::mutex xcd_mutex;
    mutable char* xcd_stream = nullptr;
    mutable XcdGeom xcd_geom{};

    ~Model() {
        if (blob) (void)hipFree(blob);
        if (xcd_stream) (void)hipFree(xcd_stream);
    }
};

static size_t align_up(size_t n, size_t a) { return (n + a - 1) / a * a; }

// Carves the weight blob and records where each file tensor goes.
static void plan_model(Model& m) {
    const Shape& s = m.shape;
    const size_t d = s.d_model, F = s.d_ff(), V = s.vocab, C = s.max_len, L = s.layers;
    size_t off = 0;
    auto take = [&](size_t n) {
        const size_t at = off;
        off = align_up(off + n, 64);  // 256-byte alignment
        return at;
    };
    std::vector<size_t> o;
    o.push_back(take(V * d));
    if (!s.modern()) o.push_back(take(C * d));
    struct LO {
        size_t wqkv, bqkv, wo, bo, w1, b1, w2, b2, g1, be1, g2, be2;
    };
    std::vector<LO> lo(L);
    for (size_t l = 0; l < L; l++) {
        lo[l].wqkv = take(3 * d * d);
        lo[l].bqkv = take(3 * d);
        lo[l].wo = take(d * d);
        lo[l].bo = take(d);
        lo[l].w1 = take((s.modern() ? 2 : 1) * F * d);
        lo[l].b1 = take(F);
        lo[l].w2 = take(d * F);
        lo[l].b2 = take(d);
        lo[l].g1 = take(d);
        lo[l].be1 = take(d);
        lo[l].g2 = take(d);
        lo[l].be2 = take(d);
    }
    const size_t ogf = take(d), obf = take(d);
    const size_t half = s.head_size() / 2;
    const size_t ocos = take(C * half + 1), osin = take(C * half + 1);
    m.blob_floats = off;
    HIP_CHECK(hipMalloc(&m.blob, off * sizeof(float)));
    HIP_CHECK(hipMemset(m.blob, 0, off * sizeof(float)));

    float* B = m.blob;
    m.E = B + o[0];
    m.P = s.modern() ? nullptr : B + o[1];
    m.place.push_back({m.E, false, 1, 0});
    if (!s.modern()) m.place.push_back({m.P, false, 1, 0});
    m.layers.resize(L);
    for (size_t l = 0; l < L; l++) {
        LayerWeights& w = m.layers[l];
        w = {B + lo[l].wqkv, B + lo[l].bqkv, B + lo[l].wo, B + lo[l].bo, B + lo[l].w1,
             B + lo[l].b1,   B + lo[l].w2,   B + lo[l].b2, B + lo[l].g1, B + lo[l].be1,
             B + lo[l].g2,   B + lo[l].be2};
        for (int q = 0; q < 3; q++) m.place.push_back({w.wqkv + q * d * d, true, 1, 0});
        m.place.push_back({w.wo, true, 1, 0});
        for (int q = 0; q < 3; q++) m.place.push_back({w.bqkv + q * d, false, 1, 0});
        m.place.push_back({w.bo, false, 1, 0});
        if (s.modern()) {
            m.place.push_back({w.w1, true, 2, 0});  // gate -> even rows
            m.place.push_back({w.w1, true, 2, 1});  // up -> odd rows
            m.place.push_back({w.w2, true, 1, 0});  // down
        } else {
            m.place.push_back({w.w1, true, 1, 0});
            m.place.push_back({w.b1, false, 1, 0});
            m.place.push_back({w.w2, true, 1, 0});
            m.place.push_back({w.b2, false, 1, 0});
        }
        m.place.push_back({w.g1, false, 1, 0});
        m.place.push_back({w.be1, false, 1, 0});
        m.place.push_back({w.g2, false, 1, 0});
        m.place.push_back({w.be2, false, 1, 0});
    }
    m.gf = B + ogf;
    m.bf = B + obf;
    m.place.push_back({m.gf, false, 1, 0});
    m.place.push_back({m.bf, false, 1, 0});
    m.rope_cos = B + ocos;
    m.rope_sin = B + osin;
}

// Shapes whose prompts go through each layer in one pass: head size 64, rows of whole
// 64-column runs (four sets of wavefronts share K in blocks of 16).
static bool rows_shape_ok(const Shape& sh) {
    return sh.head_size() == 64 && sh.d_model % 64 == 0 && sh.d_ff() % 64 == 0;
}

// Writes a split form once per model: make(blob) fills an allocation of so many bytes and says whether the weights have
// the form.  False: they have none, or there is no memory for it now (the next pass asks again).
template <class Make>
static bool make_form(SplitForm& f, size_t bytes, Make make) {
    std::lock_guard<std::mutex> lock(f.mutex);
    if (f.ready || f.unfit) return f.ready;
    DeviceBlob blob;
    if (!try_alloc(blob.at, bytes)) return false;
    if (make(blob.at)) {
        f.ready = true;
        std::swap(f.blob.at, blob.at);
    } else {
        f.unfit = true;
    }
    return f.ready;
}

// In three parts: fill calls place(src, N, K, gate_up) for every matrix and is given the place of its split form.
template <class Fill>
static bool make_split_form(SplitForm& f, size_t bytes, Fill fill) {
    return make_form(f, bytes + sizeof(int), [&](char* at) {
        int* const beyond = reinterpret_cast<int*>(at + bytes);  // set if any weight is out of range
        HIP_CHECK(hipMemset(beyond, 0, sizeof(int)));
        fill([&](const float* src, int N, int K, bool gate_up) {
            split_weights(src, N, K, gate_up, at, beyond, nullptr);
            char* const here = at;
            at += split_bytes(N, K);
            return here;
        });
        int found = 0;
        HIP_CHECK(hipMemcpy(&found, beyond, sizeof(int), hipMemcpyDeviceToHost));
        return found == 0;
    });
}

// Storage of a matrix in pairs: the blocks, its outputs' units, and the 2-norms of its rows.
struct PairPlace {
    char* w;
    float* unit;
    float* norm;
};

static size_t pair_place_bytes(size_t N, size_t K) { return pair_bytes(N, K) + 2 * pair_rows(N) * sizeof(float); }

static PairPlace place_pairs(char*& at, const float* src, int N, int K, bool gate_up) {
    PairPlace p;
    p.w = at;
    p.unit = reinterpret_cast<float*>(at + pair_bytes(N, K));
    p.norm = p.unit + pair_rows(N);
    at += pair_place_bytes(N, K);
    pair_weights(src, N, K, gate_up, p.w, p.unit, p.norm, nullptr);
    return p;
}

// Sizes of runs of values, in double.
struct Size {
    double top = 0.0, low = 0.0;
    Size(const Sizes& s) : top(s.top), low(s.low) {}
};

// The power of two that takes values of at most `bound` below 2^15, if what most of them reach, `low`, lies within 2^24 of
// it (a pair is off by 2^-51 of the bound at most); none for a bound that is no number or far from fp32's middle.
static std::optional<int> pair_exponent(double bound, double low, double room = 0x1p-24) {
    if (bound == 0.0) return 0;
    if (!(bound > 0x1p-40 && bound < 0x1p40) || !(low >= bound * room)) return std::nullopt;
    return 14 - std::ilogb(bound);
}

// Largest magnitude and largest 2-norm of a norm's rows, and what most of their values reach.
struct NormSize {
    double top, norm, low;
};

static NormSize norm_size(size_t d, const Size& g, const Size& b) {
    const double root = std::sqrt(static_cast<double>(d));
    return {root * g.top + b.top, root * (g.top + b.top), g.low};
}

// The runs of a layer's vectors and of its rows' 2-norms that bounds are made of (of a vector that the block has not, none).
enum LayerRun { RUN_WQ, RUN_WK, RUN_WV, RUN_WO, RUN_W1, RUN_W2, RUN_BQ, RUN_BK, RUN_BV, RUN_B1, RUN_G1, RUN_BE1, RUN_G2, RUN_BE2, LAYER_RUNS };
static_assert(LAYER_RUNS <= kSizeRuns, "one launch");

// The operands' powers of two, from bounds that hold for every input: a row of norm(x) has at most sqrt(d) times the
// largest gain as its largest value and as its norm (and beta), an output at most that times its row of weights, an
// average of values at most the largest of them, |gelu(z)| <= |z| and |silu(g) u| <= |g u|.  (fp32 roundings on
// the way are far from the factor of two that is left to fp16's largest number.)
static bool pair_bounds(const Shape& sh, const Sizes* run, PairLayer& l) {
    const size_t d = sh.d_model;
    const NormSize n1 = norm_size(d, run[RUN_G1], run[RUN_BE1]), n2 = norm_size(d, run[RUN_G2], run[RUN_BE2]);
    const Size wq = run[RUN_WQ], wk = run[RUN_WK], wv = run[RUN_WV], w1 = run[RUN_W1];
    const Size bq = run[RUN_BQ], bk = run[RUN_BK], bv = run[RUN_BV], b1 = run[RUN_B1];
    // (W_o and FFN2 feed no operand, but an infinite weight has no pair either)
    if (!std::isfinite(run[RUN_WO].top) || !std::isfinite(run[RUN_W2].top)) return false;
    const double query = std::sqrt(2.0) * (wq.top * n1.norm + bq.top), low_query = wq.low * n1.low;
    const double key = std::sqrt(2.0) * (wk.top * n1.norm + bk.top);  // (a rotated pair is as long as it was)
    const double value = wv.top * n1.norm + bv.top, unit = w1.top * n2.norm + b1.top;
    const double low_key = wk.low * n1.low, low_value = wv.low * n1.low, low_unit = w1.low * n2.low;
    const auto norm1 = pair_exponent(n1.top, n1.low), norm2 = pair_exponent(n2.top, n2.low);
    const auto keys = pair_exponent(key, low_key);
    const auto attn = pair_exponent(value, low_value / 64);  // (an average of many is smaller than one of them)
    const auto hidden = sh.modern() ? pair_exponent(unit * unit, low_unit * low_unit / 4) : pair_exponent(unit, low_unit / 4);
    // (A query's power of two is its own, attn_pair_kernel's, and its second part is not lifted: one power serves the whole
    // row while most of it lies within 2^16 of the largest it can hold, off by 2^-39 of that.)
    const bool queries = pair_exponent(query, low_query, 0x1p-16).has_value();
    if (!norm1 || !norm2 || !queries || !keys || !attn || !hidden) return false;
    l.norm1 = *norm1;
    l.keys = *keys;
    l.attn = *attn;
    l.norm2 = *norm2;
    l.hidden = *hidden;
    return true;
}

static bool split_layers(const Model& m) {
    const Shape& sh = m.shape;
    const int d = sh.d_model, F = sh.d_ff(), up = sh.modern() ? 2 : 1;
    const size_t per_layer = split_bytes(3 * d, d) + split_bytes(d, d) + split_bytes(up * F, d) + split_bytes(d, F);
    return make_split_form(m.layers_split, sh.layers * per_layer, [&](auto place) {
        m.split_layers.clear();
        for (const LayerWeights& w : m.layers) {
            SplitLayer l;
            l.wqkv = place(w.wqkv, 3 * d, d, false);
            l.wo = place(w.wo, d, d, false);
            l.w1 = place(w.w1, up * F, d, sh.modern());
            l.w2 = place(w.w2, d, F, false);
            m.split_layers.push_back(l);
        }
    });
}

static bool layers_in_pairs(const Model& m) {
    const Shape& sh = m.shape;
    const int d = sh.d_model, F = sh.d_ff(), up = sh.modern() ? 2 : 1;
    const size_t per_layer =
        pair_place_bytes(3 * d, d) + pair_place_bytes(d, d) + pair_place_bytes(up * F, d) + pair_place_bytes(d, F);
    const size_t sizes_at = sh.layers * per_layer;
    return make_form(m.layers_pairs, sizes_at + sh.layers * kSizeRuns * sizeof(Sizes), [&](char* at) {
        Sizes* const device = reinterpret_cast<Sizes*>(at + sizes_at);
        m.pair_layers.clear();
        for (const LayerWeights& w : m.layers) {
            const PairPlace qkv = place_pairs(at, w.wqkv, 3 * d, d, false), o = place_pairs(at, w.wo, d, d, false);
            const PairPlace ffn1 = place_pairs(at, w.w1, up * F, d, sh.modern()), ffn2 = place_pairs(at, w.w2, d, F, false);
            SizeRuns runs{};
            const auto run = [&](LayerRun r, const float* values, int n) { runs.at[r] = values, runs.n[r] = n; };
            run(RUN_WQ, qkv.norm, d), run(RUN_WK, qkv.norm + d, d), run(RUN_WV, qkv.norm + 2 * d, d);
            run(RUN_WO, o.norm, d), run(RUN_W1, ffn1.norm, up * F), run(RUN_W2, ffn2.norm, d);
            run(RUN_BQ, w.bqkv, d), run(RUN_BK, w.bqkv + d, d), run(RUN_BV, w.bqkv + 2 * d, d);
            run(RUN_G1, w.g1, d), run(RUN_G2, w.g2, d);
            if (!sh.modern()) run(RUN_B1, w.b1, F), run(RUN_BE1, w.be1, d), run(RUN_BE2, w.be2, d);
            sizes_of(runs, device + m.pair_layers.size() * kSizeRuns, nullptr);
            m.pair_layers.push_back({qkv.w, o.w, ffn1.w, ffn2.w, qkv.unit, o.unit, ffn1.unit, ffn2.unit, 0, 0, 0, 0, 0});
        }
        std::vector<Sizes> sizes(m.pair_layers.size() * kSizeRuns);
        HIP_CHECK(hipMemcpy(sizes.data(), device, sizes.size() * sizeof(Sizes), hipMemcpyDeviceToHost));
        for (size_t i = 0; i < m.pair_layers.size(); i++)
            if (!pair_bounds(sh, &sizes[i * kSizeRuns], m.pair_layers[i])) return false;
        return true;
    });
}

// The form that a pass takes: pairs (kernels_pair.h) where the model has them and they are no further from float64 than
// three parts, which a pass of the other rows takes.  Nothing else decides: what a prompt leaves must not depend on the call
// it came by, nor on what is drawn behind it.
enum SplitKind { SPLIT_NONE, SPLIT_PAIRS, SPLIT_PARTS };

static SplitKind layers_kind(const Model& m, long rows) {
    const Shape& sh = m.shape;
    const int ffn1 = (sh.modern() ? 2 : 1) * sh.d_ff();
    if (sh.d_model >= kPairMinCols && !parts_are_closer(sh.d_model, ffn1, rows) && layers_in_pairs(m)) return SPLIT_PAIRS;
    return split_layers(m) ? SPLIT_PARTS : SPLIT_NONE;
}

static SplitKind logits_kind(const Model& m, long rows) {
    const int d = m.shape.d_model, V = m.shape.vocab;
    if (d >= kPairMinCols && !logits_parts_are_closer(d, V, rows)) {
        const size_t sizes_at = pair_place_bytes(V, d);
        const bool pairs = make_form(m.logits_pairs, sizes_at + kSizeRuns * sizeof(Sizes), [&](char* at) {
            Sizes* const device = reinterpret_cast<Sizes*>(at + sizes_at);
            const PairPlace e = place_pairs(at, m.E, V, d, false);
            SizeRuns runs{{e.norm, m.gf, m.bf}, {V, d, m.shape.modern() ? 0 : d}};
            sizes_of(runs, device, nullptr);
            Sizes sizes[3];
            HIP_CHECK(hipMemcpy(sizes, device, sizeof(sizes), hipMemcpyDeviceToHost));
            const NormSize n = norm_size(d, sizes[1], sizes[2]);
            const std::optional<int> norm = pair_exponent(n.top, n.low);
            if (!norm) return false;
            m.logits_unit = e.unit;
            m.logits_norm = *norm;
            return !std::isinf(sizes[0].top);
        });
        if (pairs) return SPLIT_PAIRS;
    }
    const bool parts = make_split_form(m.logits_split, split_bytes(V, d), [&](auto place) { place(m.E, V, d, false); });
    return parts ? SPLIT_PARTS : SPLIT_NONE;
}

static std::unique_ptr<Model> upload_model(const Shape& shape, const std::vector<const float*>& t,
                                           const std::optional<Fingerprint>& fp) {
    require_gpu();
    auto m = std::make_unique<Model>();
    m->shape = shape;
    m->tokenizer = fp;
    plan_model(*m);
    const std::vector<TensorSpec> specs = tensor_specs(shape);
    if (specs.size() != t.size() || specs.size() != m->place.size())
        throw ApiError{GH_ERR_INVALID_ARGUMENT, "tensor count does not match the model shape"};

    size_t biggest = 0;
    for (size_t i = 0; i < specs.size(); i++)
        if (m->place[i].transpose)
            biggest = std::max(biggest, static_cast<size_t>(specs[i].rows) * specs[i].cols);
    float* stage = nullptr;
    HIP_CHECK(hipMalloc(&stage, std::max<size_t>(biggest, 1) * sizeof(float)));
    try {
        for (size_t i = 0; i < specs.size(); i++) {
            const size_t n = static_cast<size_t>(specs[i].rows) * specs[i].cols;
            const Placement& pl = m->place[i];
            if (!pl.transpose) {
                HIP_CHECK(hipMemcpy(pl.dst, t[i], n * sizeof(float), hipMemcpyHostToDevice));
                continue;
            }
            HIP_CHECK(hipMemcpy(stage, t[i], n * sizeof(float), hipMemcpyHostToDevice));
            const dim3 grid((specs[i].cols + 31) / 32, (specs[i].rows + 31) / 32);
            transpose_in_kernel<<<grid, dim3(32, 8)>>>(stage, specs[i].rows, specs[i].cols, pl.dst,
                                                       pl.row_mul, pl.row_off);
            HIP_CHECK(hipGetLastError());
            HIP_CHECK(hipDeviceSynchronize());
        }
    } catch (...) {
        (void)hipFree(stage);
        throw;
    }
    HIP_CHECK(hipFree(stage));

    if (shape.modern()) {
        // The rotation angles of every position, with the reference's own fp32
        // expression (inference.cpp:169-175).
        const size_t half = shape.head_size() / 2, C = shape.max_len;
        std::vector<float> cs(C * half), sn(C * half);
        for (size_t j = 0; j < half; j++) {
            const float theta = std::pow(10000.0f, -2.0f * static_cast<float>(j)
                                                       / static_cast<float>(shape.head_size()));
            for (size_t pos = 0; pos < C; pos++) {
                cs[pos * half + j] = std::cos(static_cast<float>(pos) * theta);
                sn[pos * half + j] = std::sin(static_cast<float>(pos) * theta);
            }
        }
        if (half > 0) {
            HIP_CHECK(hipMemcpy(m->rope_cos, cs.data(), cs.size() * 4, hipMemcpyHostToDevice));
            HIP_CHECK(hipMemcpy(m->rope_sin, sn.data(), sn.size() * 4, hipMemcpyHostToDevice));
        }
    }
    return m;
}

// Reads every tensor back in file layout.
static std::vector<std::vector<float>> download_model(const Model& m) {
    const std::vector<TensorSpec> specs = tensor_specs(m.shape);
    size_t biggest = 1;
    for (const TensorSpec& s : specs) biggest = std::max(biggest, static_cast<size_t>(s.rows) * s.cols);
    float* stage = nullptr;
    HIP_CHECK(hipMalloc(&stage, biggest * sizeof(float)));
    std::vector<std::vector<float>> out;
    try {
        for (size_t i = 0; i < specs.size(); i++) {
            const size_t n = static_cast<size_t>(specs[i].rows) * specs[i].cols;
            const Placement& pl = m.place[i];
            std::vector<float> host(n);
            if (!pl.transpose) {
                HIP_CHECK(hipMemcpy(host.data(), pl.dst, n * 4, hipMemcpyDeviceToHost));
            } else {
                const dim3 grid((specs[i].cols + 31) / 32, (specs[i].rows + 31) / 32);
                transpose_out_kernel<<<grid, dim3(32, 8)>>>(pl.dst, specs[i].rows, specs[i].cols,
                                                            stage, pl.row_mul, pl.row_off);
                HIP_CHECK(hipGetLastError());
                HIP_CHECK(hipMemcpy(host.data(), stage, n * 4, hipMemcpyDeviceToHost));
            }
            out.push_back(std::move(host));
        }
    } catch (...) {
        (void)hipFree(stage);
        throw;
    }
    HIP_CHECK(hipFree(stage));
    return out;
}

// ----------------------------------------------------------------- session

// What a batched step opens with: the embedding of s.tok, the greedy pick from what the last logits
// launch left and the embedding of what it picked, or nothing (the pick launch left the rows).
enum StepForm { STEP_EMBED, STEP_ARGMAX, STEP_ROWS, kStepForms };

struct Session {
    const Model* m = nullptr;
    int B = 1;
    int engine = GH_ENGINE_GRAPH;
    int page_shift = 6;
    int pages_per_seq = 0, n_pages = 0;
    int attn_chunk = 64, attn_max_chunks = 1;
    bool pick_row_in_lds = false;  // the pick's working row (vocab floats) fits in LDS beside its work area
    int work_stride = 0;           // floats per sequence of the working rows in global memory
    bool pick_global_scratch = false;
    bool use_prompt_pass = true;
    int launches_per_step = 0;

    hipStream_t stream = nullptr;
    hipGraph_t graph[kStepForms] = {};
    int form_launches[kStepForms] = {};
    hipGraphExec_t exec[kStepForms] = {};
    // Batched greedy decoding without a penalty: the logits launch leaves the largest
    // value of every run of 16 columns, and a second form of the step opens with the
    // launch that picks from those and embeds (no pick launch, no embedding launch).
    float2* best = nullptr;  // [B][best_stride]
    int best_stride = 0;
    hipEvent_t ev[3] = {nullptr, nullptr, nullptr};

    void* block = nullptr;       // the one device allocation of what a session has from the start:
    float* kv_pool = nullptr;    // everything from here to st, best, and the one-launch engine's
    int* page_table = nullptr;   // cells, xcells and ctl
    float *x = nullptr, *h = nullptr, *q = nullptr, *attn = nullptr, *hidden = nullptr,
          *logits = nullptr;
    float* work = nullptr;
    float* attn_part = nullptr;
    unsigned* attn_tickets = nullptr;
    int* tok = nullptr;   // [B] input ids of the next step
    int* hist = nullptr;  // [B][hist_stride]
    int hist_stride = 0;
    DevState* st = nullptr;
    float* uniforms = nullptr;  // device copy for generate
    size_t uniforms_cap = 0;
    float* logit_log = nullptr;  // per-step logits for gh_session_generate
    size_t logit_log_cap = 0;

    // prompt pass (all prompt tokens at once): row-major [rows][width] activations
    float *pp_x = nullptr, *pp_q = nullptr, *pp_attn = nullptr, *pp_norm = nullptr, *pp_hidden = nullptr;
    char *pp_split = nullptr, *pp_split_hidden = nullptr;  // split rows of d_model and of d_ff columns
    size_t pp_rows = 0;
    char* pp_kv = nullptr;  // split keys and values of the layer at hand
    size_t pp_kv_bytes = 0;
    float* pp_part = nullptr;  // partial attention results
    size_t pp_part_floats = 0;
    int* score_targets = nullptr;  // [B][length] of the scored tokens, and
    float* score_nll = nullptr;    // what they cost
    size_t score_cap = 0;
    float2* nll_part = nullptr;  // [pp_rows][split_nll_stride(vocab)] of rows being scored
    float* nll_target = nullptr;  // [pp_rows]
    size_t nll_rows = 0;

    // persistent engine
    Cell* cells = nullptr;  // xa, xb, q, kn, vn, at (d each), hid (F), token (1)
    size_t cells_count = 0;
    PersistCtl* ctl = nullptr;
    unsigned epoch = 1;         // tag base; grows with every step, never reused
    unsigned arrive_total = 0;  // logits phases completed so far
    int persist_grid = 0;
    unsigned long long* prof = nullptr;  // phase timestamps when GRADHIP_PROF_DUMP is set
    int prof_cap = 0;
    size_t persist_lds = 0;
    // ... its XCD-sharded form (kernels_xcd.h)
    bool xcd = false;         // the kernel and its buffers are ready
    bool xcd_row_lds = false;
    bool row_picks_only = false;  // GH_FLAG_ROW_PICKS
    Cell* xcells = nullptr;
    unsigned xcd_cells_count = 0;
    unsigned xcd_launches = 0;
    unsigned xcd_ring_units = 0, xcd_ring_units_wg0 = 0;
    size_t xcd_lds = 0;
    bool xcd_all_slices = false;  // every workgroup of an XCD takes a slice of the attention at any context

    // steps of a few sequences as one launch for all layers (kernels_resident.h)
    bool resident = false;  // ... is built for this session
    Cell* rcells = nullptr;
    size_t rcells_count = 0;
    ResidentCtl* rctl = nullptr;
    unsigned repoch = 1;    // tag base; grows with every launch, re-based by clearing the cells
    unsigned rspin_limit = 1u << 18;
    int impatient_from = 0, impatient_n = 0;  // (tests: launches that have spins_impatient looks instead)
    unsigned spins_impatient = 0;
    int resident_launches = 0;   // resident launches made so far
    bool resident_off = false;   // the rest of this call runs as launches
    int resident_backoff = 1 << 12;  // steps that run as launches behind the next step that gives up
    std::unique_lock<std::mutex> resident_lock;  // this call's hold on g_persist_gate
    int resident_rest = 0;   // steps to run as launches before the gate is tried again
    int resident_ahead = 0;  // resident steps enqueued since the last of window_ev was recorded
    int resident_window = 0; // how often that was, in this hold
    hipEvent_t window_ev[2] = {nullptr, nullptr};
    // what is on the stream in front of the next step and may take long: nothing, all of it, or up to ev[1]
    enum { AHEAD_NONE, AHEAD_STREAM, AHEAD_PROMPT } ahead = AHEAD_NONE;
    float* start_logits = nullptr;  // a copy of the logits that a run of steps began with

    void* host_block = nullptr;    // one pinned allocation, which kernels read and write directly:
    float* host_logits = nullptr;  // B * V
    int* host_ids = nullptr;       // [2][B * hist_stride] ids on their way to or from the device
    int* host_err = nullptr;       // landing spot for the device error flag
    // streaming from the persistent kernel
    unsigned long long* feed = nullptr;  // [hist_stride] {token, tag} per pick of a launch
    unsigned* stop_word = nullptr;       // set by the host to end a run at the next pick
    unsigned feed_base = 0;              // tags of a launch are feed_base + 1 ...; never reused

    int pos = 0;     // host mirror of DevState
    int n_hist = 0;
    int picks = 0;
    gh_timing timing{};

    ~Session() {
#ifdef GH_PICK_TICKS
        {
            unsigned long long t[32] = {};
            if (read_pick_ticks(t)) {
                std::fprintf(stderr, "pick ticks (10 ns, summed):");
                for (unsigned long long v : t) std::fprintf(stderr, " %llu", v);
                std::fprintf(stderr, "\n");
            }
        }
#endif
        if (prof) {
            // Developer aid: phase-end timestamps of the last persistent launch.
            std::vector<unsigned long long> host(prof_cap);
            if (hipMemcpy(host.data(), prof, host.size() * 8, hipMemcpyDeviceToHost) == hipSuccess) {
                if (std::FILE* f = std::fopen(std::getenv("GRADHIP_PROF_DUMP"), "w")) {
                    for (size_t i = 0; i < host.size() / 2 && host[i]; i++) std::fprintf(f, "%llu\n", host[i]);
                    std::fprintf(f, "0\n");
                    for (size_t i = host.size() / 2; i + 3 < host.size() - 112 && host[i]; i += 4)
                        std::fprintf(f, "%llu\n%llu\n%llu\n", host[i + 2], host[i], host[i + 1]);
                    std::fprintf(f, "0\n");
                    for (size_t i = host.size() - 112; i < host.size(); i++) std::fprintf(f, "%llu\n", host[i]);
                    std::fclose(f);
                }
            }
            (void)hipFree(prof);
        }
        for (hipGraphExec_t e : exec)
            if (e) (void)hipGraphExecDestroy(e);
        for (hipGraph_t g : graph)
            if (g) (void)hipGraphDestroy(g);
        for (hipEvent_t e : {ev[0], ev[1], ev[2], window_ev[0], window_ev[1]})
            if (e) (void)hipEventDestroy(e);
        for (void* p : {block, static_cast<void*>(uniforms), static_cast<void*>(logit_log),
                        static_cast<void*>(pp_x), static_cast<void*>(pp_q), static_cast<void*>(pp_attn),
                        static_cast<void*>(pp_norm), static_cast<void*>(pp_hidden), static_cast<void*>(pp_split),
                        static_cast<void*>(pp_split_hidden), static_cast<void*>(pp_kv), static_cast<void*>(pp_part),
                        static_cast<void*>(score_targets), static_cast<void*>(score_nll),
                        static_cast<void*>(nll_part), static_cast<void*>(nll_target), static_cast<void*>(start_logits)})
            if (p) (void)hipFree(p);
        if (host_block) (void)hipHostFree(host_block);
        if (stream) (void)hipStreamDestroy(stream);
    }
};

// The persistent kernel's workgroups wait for one another, so all of them have to
// be resident at once: one per compute unit.  Two such launches in flight at the
// same time (two sessions on two host threads) could each hold a part of the
// GPU and wait for the rest for ever.  Every entry point that launches the
// kernel therefore holds this process-wide lock from before the launch until
// the stream has been synchronised.  Sessions whose steps may be resident take it when it is free and
// somebody does not want it (resident_begin); the others never do.
static std::mutex g_persist_gate;
static std::atomic<int> g_gate_waiting{0};  // calls of the one-launch engine that are waiting for it

static thread_local int g_gate_depth = 0;

struct PersistGate {
    std::unique_lock<std::mutex> lock;
    explicit PersistGate(const struct Session& s);
    ~PersistGate() {
        if (lock.owns_lock()) g_gate_depth--;
    }
    PersistGate(const PersistGate&) = delete;
    PersistGate& operator=(const PersistGate&) = delete;
};

PersistGate::PersistGate(const Session& s) {
    if (s.engine != GH_ENGINE_PERSISTENT) return;
    // a stream callback that calls into another persistent session would wait for itself
    if (g_gate_depth > 0)
        throw ApiError{GH_ERR_RUNTIME, "a persistent-engine call is already running on this thread "
                                       "(token callbacks must not call into persistent-engine sessions)"};
    g_gate_waiting.fetch_add(1);
    lock = std::unique_lock<std::mutex>(g_persist_gate);
    g_gate_waiting.fetch_sub(1);
    g_gate_depth++;
}

static KvLayout kv_layout(const Session& s) {
    return KvLayout{s.kv_pool,         s.page_table,           s.n_pages, s.pages_per_seq,
                    s.m->shape.heads,  s.m->shape.head_size(), s.page_shift};
}

template <typename T>
static void dev_alloc(T*& p, size_t n) {
    HIP_CHECK(hipMalloc(&p, std::max<size_t>(n, 1) * sizeof(T)));
    HIP_CHECK(hipMemset(p, 0, std::max<size_t>(n, 1) * sizeof(T)));
}

// Several arrays in one allocation, each on a boundary of 256 bytes: a session has some twenty,
// and allocating, clearing and freeing them one by one was most of the 375 us that creating and
// destroying it took.
struct Block {
    struct Part {
        void* at;  // T**
        size_t offset;
    };
    std::vector<Part> parts;
    size_t bytes = 0;
    template <typename T>
    void add(T*& p, size_t n) {
        parts.push_back({static_cast<void*>(&p), bytes});
        bytes += (std::max<size_t>(n, 1) * sizeof(T) + 255) / 256 * 256;
    }
    void place(void* base) const {
        for (const Part& part : parts) {
            void* p = static_cast<char*>(base) + part.offset;
            std::memcpy(part.at, &p, sizeof(p));
        }
    }
};

// ---- kernel dispatch

template <int PRO, int EPI>
static void launch_gemv(const GemvParams& p, int batch, hipStream_t st) {
    const int K = p.K;
    const bool aligned = (K % 256 == 0) && (p.in_stride % 4 == 0);
    const int kv = aligned ? K / 256 : 0;
    auto go = [&](auto kernel, int rows_per_wave) {
        const int waves = (p.N + rows_per_wave - 1) / rows_per_wave;
        const dim3 grid((waves + 3) / 4, batch);
        enqueue(kernel, grid, dim3(256), 0, st, p);
    };
    switch (kv) {
        case 1: go(gemv_kernel<1, 2, PRO, EPI>, 4); break;
        case 2: go(gemv_kernel<2, 2, PRO, EPI>, 4); break;
        case 3: go(gemv_kernel<3, 2, PRO, EPI>, 4); break;
        case 4: go(gemv_kernel<4, 2, PRO, EPI>, 4); break;
        case 8: go(gemv_kernel<8, 1, PRO, EPI>, 2); break;
        case 12: go(gemv_kernel<12, 1, PRO, EPI>, 2); break;
        default: go(gemv_kernel<0, 1, PRO, EPI>, 2); break;
    }
    HIP_CHECK(hipGetLastError());
}

static void launch_attn(const AttnParams& p, int batch, hipStream_t st) {
    const int hs = p.kv.head_size;
    const dim3 grid(p.max_chunks, p.kv.heads, batch);
    if (hs == 64) {
        if (p.kv.page_shift >= 5 && p.chunk % 128 == 0)
            enqueue(attn_decode64_kernel<true>, grid, dim3(256), 0, st, p);
        else
            enqueue(attn_decode64_kernel<false>, grid, dim3(256), 0, st, p);
        HIP_CHECK(hipGetLastError());
        return;
    }
    const size_t lds = (static_cast<size_t>(p.chunk) + 4 * hs + 8) * sizeof(float);
    switch (hs) {
        case 8: enqueue(attn_decode_kernel<8>, grid, dim3(256), lds, st, p); break;
        case 16: enqueue(attn_decode_kernel<16>, grid, dim3(256), lds, st, p); break;
        case 32: enqueue(attn_decode_kernel<32>, grid, dim3(256), lds, st, p); break;
        case 64: enqueue(attn_decode_kernel<64>, grid, dim3(256), lds, st, p); break;
        case 128: enqueue(attn_decode_kernel<128>, grid, dim3(256), lds, st, p); break;
        default: enqueue(attn_decode_kernel<0>, grid, dim3(256), lds, st, p); break;
    }
    HIP_CHECK(hipGetLastError());
}

// Batches of this size and up go to the matrix cores.
constexpr int kMinGemmBatch = 2;

// One projection with its fused prologue / epilogue; returns the launches made.
template <int PRO, int EPI>
static int project(Session& s, GemvParams g, hipStream_t st) {
    const int B = s.B;
    if (B >= kMinGemmBatch && gemm_shape_ok(g.K, g.in_stride)) {
        if (PRO == PRO_RMSNORM) {
            // the norm rides inside the projection
            launch_gemm16<EPI, true>(g, B, st);
            HIP_CHECK(hipGetLastError());
            return 1;
        }
        int launches = 1;
        if (PRO != PRO_PLAIN) {
            launch_layernorm_rows(g.in, g.gamma, g.beta, s.h, B, g.K, st);
            HIP_CHECK(hipGetLastError());
            g.in = s.h;
            g.in_stride = g.K;
            launches++;
        }
        launch_gemm16<EPI, false>(g, B, st);
        HIP_CHECK(hipGetLastError());
        return launches;
    }
    launch_gemv<PRO, EPI>(g, B, st);
    return 1;
}

// final norm -> logits = h @ E^T (inference.cpp:251-254) from the rows in s.x
// advance: the launch also ends the step (pos_++).
static int enqueue_logits(Session& s, bool advance) {
    const Model& m = *s.m;
    const Shape& sh = m.shape;
    const bool modern = sh.modern();
    GemvParams g{};
    g.W = m.E;
    g.bias = nullptr;
    g.N = sh.vocab;
    g.K = sh.d_model;
    g.in = s.x;
    g.in_stride = sh.d_model;
    g.gamma = m.gf;
    g.beta = m.bf;
    g.out = s.logits;
    g.out_stride = sh.vocab;
    g.advance = advance ? s.st : nullptr;
    g.best = s.best;
    g.best_stride = s.best_stride;
    return modern ? project<PRO_RMSNORM, EPI_STORE>(s, g, s.stream)
                  : project<PRO_LAYERNORM, EPI_STORE>(s, g, s.stream);
}

// One layer of a step for every sequence, on the rows in s.x at the position in s.st.
// query_only: the position's key and value are in the cache already.
static int enqueue_layer(Session& s, int l, bool query_only) {
    const Model& m = *s.m;
    const Shape& sh = m.shape;
    const int d = sh.d_model, F = sh.d_ff(), B = s.B;
    const bool modern = sh.modern();
    hipStream_t st = s.stream;
    int launches = 0;

    // What a projection launch touches into the L2s for the projection after it (NextWeights):
    // the whole matrix, in the 16-row tiles that launch reads it in; up to 48 sequences.
    const bool touch = B >= kMinGemmBatch && B <= 48;
    const auto next_matrix = [&](const float* W, int N, int K) {
        NextWeights f{};
        if (!touch || !gemm_shape_ok(K, K) || N % 16 != 0) return f;
        f.base = W;
        f.chunk_lines = K / 2;  // 16 rows of K floats
        f.chunks = N / 16;
        const long long lines = static_cast<long long>(f.chunks) * f.chunk_lines;
        f.blocks = static_cast<int>(std::min<long long>(128, (lines + 8191) / 8192 * 8));  // up to four lines per thread of 256
        return f;
    };

    const LayerWeights& w = m.layers[l];
    GemvParams g{};
    g.kv = kv_layout(s);
    g.layer = l;
    g.d_model = d;
    g.st = s.st;

    // norm1 -> fused Q,K,V projection (+bias, RoPE) -> q buffer / cache row
    g.W = w.wqkv;
    g.bias = w.bqkv;
    g.N = query_only ? d : 3 * d;
    g.K = d;
    g.in = s.x;
    g.in_stride = d;
    g.gamma = w.g1;
    g.beta = w.be1;
    g.out = s.q;
    g.out_stride = d;
    g.rope = modern;
    g.rope_cos = m.rope_cos;
    g.rope_sin = m.rope_sin;
    g.next = NextWeights{};  // attention follows
    launches += modern ? project<PRO_RMSNORM, EPI_QKV>(s, g, st)
                       : project<PRO_LAYERNORM, EPI_QKV>(s, g, st);

    AttnParams a{};
    a.q = s.q;
    a.out = s.attn;
    a.kv = g.kv;
    a.layer = l;
    a.d_model = d;
    a.st = s.st;
    a.chunk = s.attn_chunk;
    a.max_chunks = s.attn_max_chunks;
    a.scale = 1.0f / std::sqrt(static_cast<float>(sh.head_size()));
    a.part = s.attn_part;
    a.tickets = s.attn_tickets;
    launch_attn(a, B, st);
    launches++;

    // x += b_o + attn @ W_o
    g.W = w.wo;
    g.bias = w.bo;
    g.N = d;
    g.K = d;
    g.in = s.attn;
    g.in_stride = d;
    g.out = s.x;
    g.out_stride = d;
    g.next = next_matrix(w.w1, modern ? 2 * F : F, d);
    launches += project<PRO_PLAIN, EPI_RESID>(s, g, st);

    // norm2 -> FFN
    g.in = s.x;
    g.in_stride = d;
    g.gamma = w.g2;
    g.beta = w.be2;
    g.out = s.hidden;
    g.out_stride = F;
    g.W = w.w1;
    g.K = d;
    g.next = next_matrix(w.w2, d, F);
    if (modern) {
        g.bias = nullptr;
        g.N = 2 * F;
        launches += project<PRO_RMSNORM, EPI_SWIGLU>(s, g, st);
    } else {
        g.bias = w.b1;
        g.N = F;
        launches += project<PRO_LAYERNORM, EPI_GELU>(s, g, st);
    }
    g.W = w.w2;
    g.bias = modern ? nullptr : w.b2;
    g.N = d;
    g.K = F;
    g.in = s.hidden;
    g.in_stride = F;
    g.out = s.x;
    g.out_stride = d;
    g.next = l + 1 < sh.layers ? next_matrix(m.layers[l + 1].wqkv, 3 * d, d) : NextWeights{};
    launches += project<PRO_PLAIN, EPI_RESID>(s, g, st);
    return launches;
}

// ---- all layers of a step in one launch (kernels_resident.h)

// A call whose steps are resident enqueues them far ahead of the GPU, and whoever waits for the gate can have it only
// when what is enqueued has run.  So no more than two windows of steps are, and a hold begins when what may take
// long in front of it (a prompt, steps as launches) is done: a call on the one-launch engine waits for at most 2 x 8
// steps. (One step of a single sequence beside 13 sequences x 600 tokens: 133 ms before there were windows, 2.9 at
// most with them; beside 16 x 400 behind 1500 positions 189, 6.9. Alone, 48 tokens of 13 sequences 10.76 ms either
// way, 16 behind 1536 positions 35.47.)
constexpr int kResidentWindow = 8;
// Steps as launches behind a hold that was given up to somebody, about what the call got that waited for it.
constexpr int kResidentRest = 64;

// The stream has been synchronised (or nothing resident is on it).
static void resident_end(Session& s) {
    s.ahead = Session::AHEAD_NONE;
    s.resident_ahead = s.resident_window = 0;
    if (!s.resident_lock.owns_lock()) return;
    g_gate_depth--;
    s.resident_lock.unlock();
    s.resident_lock = {};
}

// What this call launches may take the whole GPU from here on: the gate that resident launches share is this
// session's until resident_end. False, and the step runs as a launch per operation, when another
// session has it or waits for it or this thread is inside a callback of one that does: both forms give the same bits.
static bool resident_begin(Session& s) {
    if (s.resident_lock.owns_lock()) {
        if (g_gate_waiting.load(std::memory_order_relaxed) == 0) return true;
        HIP_CHECK(hipStreamSynchronize(s.stream));
        resident_end(s);
        s.resident_rest = kResidentRest;
        return false;
    }
    if (s.resident_rest > 0) {
        s.resident_rest--;
        return false;
    }
    if (g_gate_depth > 0 || g_gate_waiting.load(std::memory_order_relaxed) != 0) return false;
    std::unique_lock<std::mutex> lock(g_persist_gate, std::try_to_lock);
    if (!lock.owns_lock()) return false;
    if (s.ahead != Session::AHEAD_NONE) {
        lock.unlock();
        HIP_CHECK(s.ahead == Session::AHEAD_PROMPT ? hipEventSynchronize(s.ev[1]) : hipStreamSynchronize(s.stream));
        s.ahead = Session::AHEAD_NONE;
        if (!lock.try_lock()) return false;
    }
    s.resident_lock = std::move(lock);
    g_gate_depth++;
    return true;
}

// Behind a resident step: waits until the window before the present one has run.
static void resident_pace(Session& s) {
    if (++s.resident_ahead < kResidentWindow) return;
    s.resident_ahead = 0;
    HIP_CHECK(hipEventRecord(s.window_ev[s.resident_window & 1], s.stream));
    if (s.resident_window++ > 0) HIP_CHECK(hipEventSynchronize(s.window_ev[s.resident_window & 1]));
}

// Ends the call's hold however the call ends; what it launched has left the GPU by then.
struct ResidentScope {
    Session& s;
    const int exceptions = std::uncaught_exceptions();
    explicit ResidentScope(Session& session) : s(session) {}
    ~ResidentScope() {
        if (std::uncaught_exceptions() > exceptions && s.resident_lock.owns_lock()) (void)hipStreamSynchronize(s.stream);
        resident_end(s);
        s.resident_off = false;
    }
    ResidentScope(const ResidentScope&) = delete;
    ResidentScope& operator=(const ResidentScope&) = delete;
};

// (sequence, head, run of positions): what the attention of the next step consists of.
static int resident_items(const Session& s) { return s.B * s.m->shape.heads * (s.pos / s.attn_chunk + 1); }

// For the next step of this session: can and may it run that way?
static bool resident_now(Session& s) {
    if (!s.resident || s.resident_off) return false;
    if (!resident_kernel_for(s.m->shape, s.B, resident_items(s))) {
        if (s.resident_lock.owns_lock()) {  // (the context has outgrown the kernel)
            HIP_CHECK(hipStreamSynchronize(s.stream));
            resident_end(s);
        }
        return false;
    }
    return resident_begin(s);
}

static void launch_resident(Session& s) {
    const Model& m = *s.m;
    const Shape& sh = m.shape;
    // Tags are matched by equality and must not come round to one a stale cell holds.
    if ((static_cast<unsigned long long>(s.repoch) + 2ull * sh.layers + 2ull) * 8ull >= 0xF0000000ull) {
        HIP_CHECK(hipMemsetAsync(s.rcells, 0, s.rcells_count * sizeof(Cell), s.stream));
        s.repoch = 1;
    }
    ResidentParams p{};
    p.layer0 = m.layers[0].wqkv;
    p.rope_cos = m.rope_cos;
    p.rope_sin = m.rope_sin;
    p.x = s.x;
    p.kv = kv_layout(s);
    p.cells = s.rcells;
    p.ctl = s.rctl;
    p.B = s.B;
    p.L = sh.layers;
    p.pos = s.pos;
    p.chunk = s.attn_chunk;
    p.epoch = s.repoch;
    const int launch = s.resident_launches;
    s.resident_launches = launch < INT_MAX ? launch + 1 : launch;
    p.spin_limit = launch >= s.impatient_from && launch - s.impatient_from < s.impatient_n ? s.spins_impatient : s.rspin_limit;
    s.repoch += static_cast<unsigned>(sh.layers);
    hipLaunchKernelGGL(resident_kernel_for(sh, s.B, resident_items(s)), dim3(kResidentGrid), dim3(kResidentThreads),
                       static_cast<size_t>(s.B) * s.pages_per_seq * sizeof(int), s.stream, p);
    HIP_CHECK(hipGetLastError());
}

// One InferenceSession::step for every sequence (inference.cpp:150-258),
// enqueued on the session stream.  Returns the number of launches.
// resident: all layers in one launch.
static int enqueue_step(Session& s, StepForm form, bool resident = false) {
    const Model& m = *s.m;
    const Shape& sh = m.shape;
    const int d = sh.d_model, B = s.B;
    hipStream_t st = s.stream;
    int launches = 0;

    if (form == STEP_ARGMAX) {
        // text_gen.cpp:52-60
        enqueue(argmax_embed_kernel, dim3(B), dim3(kArgmaxThreads), 0, st, s.best, s.best_stride, s.st, s.hist,
                s.hist_stride, s.tok, m.E, m.P, s.x, d);
    } else if (form == STEP_EMBED) {
        enqueue(embed_kernel, dim3((d + 255) / 256, B), dim3(256), 0, st, m.E, m.P, s.tok, s.st, s.x, d);
    }
    HIP_CHECK(hipGetLastError());
    launches += form != STEP_ROWS;

    if (resident) {
        launch_resident(s);
        launches++;
    } else {
        for (int l = 0; l < sh.layers; l++) launches += enqueue_layer(s, l, /*query_only=*/false);
    }
    launches += enqueue_logits(s, /*advance=*/true);
    return launches;
}

// ---- persistent engine

// ---- the XCD-sharded form of the persistent kernel (kernels_xcd.h)

// The XCD-sharded kernel runs only where GH_FLAG_XCD_PERSISTENT asks for it.  It used to
// be the default for launches that start at position 1024 or later, where it spreads a
// head's context over the workgroups of an XCD; since the all-to-all kernel shares a
// head's long context among idle workgroups itself it is the faster one at every
// position.  Per token on one box, Llama block d768 L8 V16000, greedy, XCD-sharded /
// all-to-all: positions 256..512 168 / 132, 512..768 178 / 144, 1024..1280 196 / 149,
// 2048..2304 228 / 156, 3072..3328 259 / 160, 3800..4056 277 / 162.

// Splits the model over eight XCDs: heads g and g + 8, and a run of hidden units
// sized so that every XCD streams about the same number of bytes per layer.
// False when the kernel's split does not fit the shape.
static bool xcd_geometry(const Shape& sh, XcdGeom& gm) {
    if (!xcd_kernel_for(sh, true, false)) return false;
    const int D = sh.d_model, F = sh.d_ff(), H = sh.heads;
    if (H < kXcds || H > 2 * kXcds || F % 4 != 0 || sh.layers < 1 || sh.max_len > 4096) return false;
    gm = XcdGeom{};
    gm.D = D;
    gm.F = F;
    gm.V = sh.vocab;
    gm.L = sh.layers;
    gm.H = H;
    const double per_head = 4.0 * 64.0 * D, per_unit = 3.0 * D;
    const double target = (H * per_head + F * per_unit) / kXcds;
    double want_sum = 0.0;
    int at = 0;
    for (int g = 0; g < kXcds; g++) {
        XcdShard& x = gm.shard[g];
        x.nh = g + kXcds < H ? 2 : 1;
        x.head[0] = g;
        x.head[1] = g + kXcds < H ? g + kXcds : g;
        want_sum += (target - x.nh * per_head) / per_unit;
        int end = g == kXcds - 1 ? F : static_cast<int>(std::lround(want_sum / 4.0)) * 4;
        end = std::min(std::max(end, at), F);
        x.u0 = at;
        x.nu = end - at;
        at = end;
        if (x.nu < kWgPerXcd || x.nu > 512) return false;  // every workgroup owns a unit; the XCD's units fit the LDS row
    }
    unsigned stride = 0;
    for (int g = 0; g < kXcds; g++)
        for (int r = 0; r < kWgPerXcd; r++) {
            const XcdWg w = xcd_wg(gm, g, r);
            if (w.nu < 1 || w.nu > kXcdMaxUnitsPerWg) return false;
            stride = std::max(stride, w.layers_units + w.logits_units);
        }
    gm.stride_units = stride;
    return true;
}

// One block of a weight matrix on its way into a workgroup's stream: rows x cols
// floats from blob[src + row * src_ld] to stream[dst + row * dst_ld], each column
// multiplied by a norm gain when gamma >= 0 (the gain of the norm in front of the
// product is folded into the weights: (g * x) . w == x . (g * w)).
struct XcdCopy {
    unsigned long long dst, src;
    long long gamma;
    int rows, cols, src_ld, dst_ld;
};

__global__ void xcd_copy_kernel(const XcdCopy* list, const float* __restrict__ blob, float* __restrict__ out) {
    const XcdCopy c = list[blockIdx.x];
    const int n = c.rows * c.cols;
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
        const int row = i / c.cols, col = i - row * c.cols;
        float v = blob[c.src + static_cast<size_t>(row) * c.src_ld + col];
        if (c.gamma >= 0) v *= blob[c.gamma + col];
        out[c.dst + static_cast<size_t>(row) * c.dst_ld + col] = v;
    }
}

// Builds the per-workgroup weight streams of a model (once).
static void xcd_build_stream(const Model& m) {
    std::lock_guard<std::mutex> lock(m.xcd_mutex);
    if (m.xcd_stream) return;
    XcdGeom gm;
    if (!xcd_geometry(m.shape, gm)) throw ApiError{GH_ERR_RUNTIME, "no XCD split for this model shape"};
    const size_t D = gm.D, F = gm.F, RW = D / kWgPerXcd;
    const size_t stride_floats = static_cast<size_t>(gm.stride_units) * kXcdUnit / 4;
    auto at = [&](const float* ptr) { return static_cast<unsigned long long>(ptr - m.blob); };
    std::vector<XcdCopy> list;
    for (int g = 0; g < kXcds; g++)
        for (int r = 0; r < kWgPerXcd; r++) {
            const XcdWg w = xcd_wg(gm, g, r);
            const XcdShard& sh = gm.shard[g];
            const size_t base = static_cast<size_t>(g * kWgPerXcd + r) * stride_floats;
            for (int l = 0; l < gm.L; l++) {
                const LayerWeights& lw = m.layers[l];
                const size_t lb = base + static_cast<size_t>(l) * (w.layer_bytes / 4);
                // pairs of Q / K / V rows: pair i of the XCD is (head slot, section, j)
                for (int q = 0; q < w.ppw; q++) {
                    const int pi = r * w.ppw + q, hi = pi / 96, rem = pi % 96, sec = rem / 32, j = rem % 32;
                    const size_t row = static_cast<size_t>(sec) * D + static_cast<size_t>(sh.head[hi]) * 64 + 2 * j;
                    const size_t pb = lb + static_cast<size_t>(q) * (w.pair_bytes / 4);
                    list.push_back({pb, at(lw.wqkv) + row * D, static_cast<long long>(at(lw.g1)), 2,
                                    static_cast<int>(D), static_cast<int>(D), static_cast<int>(D)});
                    list.push_back({pb + 2 * D, at(lw.bqkv) + row, -1, 1, 2, 2, 2});
                }
                // W_o: this workgroup's rows, the columns of the XCD's heads
                for (int hi = 0; hi < w.nh; hi++)
                    list.push_back({lb + w.o_wo / 4 + static_cast<size_t>(hi) * 64,
                                    at(lw.wo) + (static_cast<size_t>(r) * RW) * D + static_cast<size_t>(sh.head[hi]) * 64,
                                    -1, static_cast<int>(RW), 64, static_cast<int>(D), w.KC});
                list.push_back({lb + w.o_bo / 4, at(lw.bo) + static_cast<size_t>(r) * RW, -1, 1, static_cast<int>(RW),
                                static_cast<int>(RW), static_cast<int>(RW)});
                // gate and up rows of this workgroup's hidden units (row 2u gate, 2u + 1 up)
                list.push_back({lb + w.o_gu / 4, at(lw.w1) + static_cast<size_t>(2 * w.ub) * D,
                                static_cast<long long>(at(lw.g2)), 2 * w.nu, static_cast<int>(D),
                                static_cast<int>(D), static_cast<int>(D)});
                // W_down: this workgroup's rows, the columns of the XCD's hidden units
                list.push_back({lb + w.o_dn / 4, at(lw.w2) + (static_cast<size_t>(r) * RW) * F + static_cast<size_t>(w.u0),
                                -1, static_cast<int>(RW), w.UG, static_cast<int>(F), w.UG});
            }
            // its rows of the logits matrix, with the final norm's gain
            if (w.nrows > 0)
                list.push_back({base + static_cast<size_t>(w.layers_units) * kXcdUnit / 4,
                                at(m.E) + static_cast<size_t>(w.v0) * D, static_cast<long long>(at(m.gf)), w.nrows,
                                static_cast<int>(D), static_cast<int>(D), static_cast<int>(D)});
        }
    const size_t total = static_cast<size_t>(kXcds * kWgPerXcd) * stride_floats;
    char* stream = nullptr;
    XcdCopy* dlist = nullptr;
    HIP_CHECK(hipMalloc(&stream, total * sizeof(float)));
    try {
        HIP_CHECK(hipMemset(stream, 0, total * sizeof(float)));
        HIP_CHECK(hipMalloc(&dlist, list.size() * sizeof(XcdCopy)));
        HIP_CHECK(hipMemcpy(dlist, list.data(), list.size() * sizeof(XcdCopy), hipMemcpyHostToDevice));
        hipLaunchKernelGGL(xcd_copy_kernel, dim3(static_cast<unsigned>(list.size())), dim3(256), 0, nullptr, dlist,
                           m.blob, reinterpret_cast<float*>(stream));
        HIP_CHECK(hipGetLastError());
        HIP_CHECK(hipDeviceSynchronize());
    } catch (...) {
        if (dlist) (void)hipFree(dlist);
        (void)hipFree(stream);
        throw;
    }
    HIP_CHECK(hipFree(dlist));
    m.xcd_geom = gm;
    m.xcd_stream = stream;
}

// The one-launch kernels find a layer's tensors by address arithmetic (layer_at): they must
// follow each other without gaps, layer after layer.
static bool layers_back_to_back(const Model& m) {
    const Shape& sh = m.shape;
    const size_t d = sh.d_model, F = sh.d_ff();
    const size_t per_layer = layer_floats(d, F, sh.modern());
    const float* base = m.layers[0].wqkv;
    for (size_t l = 0; l < m.layers.size(); l++) {
        const LayerWeights& w = m.layers[l];
        const float* b = base + l * per_layer;
        const float* want[12];
        size_t i = 0;
        for (const size_t n : {3 * d * d, 3 * d, d * d, d, (sh.modern() ? 2 : 1) * F * d, F, d * F, d, d, d, d, d}) {
            want[i++] = b;
            b += n;
        }
        const float* have[12] = {w.wqkv, w.bqkv, w.wo, w.bo, w.w1, w.b1, w.w2, w.b2, w.g1, w.be1, w.g2, w.be2};
        for (i = 0; i < 12; i++)
            if (have[i] != want[i]) return false;
    }
    return true;
}

static const char* persist_unavailable(const Session& s, int lds_bytes, int cus) {
    const Shape& sh = s.m->shape;
    if (s.B != 1) return "the persistent engine decodes one sequence";
    if (!persist_kernel_for(sh, s.pick_row_in_lds)) return "the persistent engine has no kernel for this model shape";
    if (sh.max_len > 4096) return "the persistent engine handles contexts up to 4096";
    if (cus < sh.heads) return "the GPU has fewer compute units than the model has heads";
    (void)lds_bytes;
    if (!layers_back_to_back(*s.m)) return "the persistent engine needs the layers' tensors back to back";
    return nullptr;
}

// One launch: n_prompt steps fed from the history, then rounds of pick + step.
// feed: the kernel reports every pick in the session's pinned feed and honours its
// stop word and stop_token.
static void persist_run(Session& s, int n_prompt, int n_steps, int n_picks, bool start_with_pick,
                        const gh_sampling* o, const float* dev_uniforms, int u_stride, uint64_t seed,
                        float* logit_log, bool feed = false, int stop_token = -1, int tok0 = -1) {
    const Model& m = *s.m;
    const Shape& sh = m.shape;
    if (n_steps <= 0 && n_picks <= 0) return;
    // Tags are (epoch + step) * (layers + 1) * 8 + phase in 32 bits and are matched by
    // equality, so they must not come round to a value a stale cell may still hold:
    // long before that the cells are cleared on the stream (tag 0 is never used) and
    // the epoch starts over.  Arrival counts are compared by wrap-safe difference.
    {
        const unsigned long long per_step = static_cast<unsigned long long>(sh.layers + 1) * 8ull;
        const unsigned long long last = (static_cast<unsigned long long>(s.epoch) + n_steps + 2ull) * per_step + 8ull;
        if (last >= 0xF0000000ull) {
            HIP_CHECK(hipMemsetAsync(s.cells, 0, s.cells_count * sizeof(Cell), s.stream));
            if (s.xcells) HIP_CHECK(hipMemsetAsync(s.xcells, 0, s.xcd_cells_count * sizeof(Cell), s.stream));
            s.epoch = 1;
        }
    }
    PersistParams p{};
    p.E = m.E;
    p.P = m.P;
    p.layer0 = m.layers[0].wqkv;
    p.gf = m.gf;
    p.bf = m.bf;
    p.rope_cos = m.rope_cos;
    p.rope_sin = m.rope_sin;
    p.d = sh.d_model;
    p.F = sh.d_ff();
    p.V = sh.vocab;
    p.L = sh.layers;
    p.H = sh.heads;
    p.kv = kv_layout(s);
    p.cells = s.cells;
    p.logits = s.logits;
    p.logit_log = logit_log;
    p.ctl = s.ctl;
    p.hist = s.hist;
    p.pos0 = s.pos;
    p.n_prompt = n_prompt;
    p.n_steps = n_steps;
    p.n_picks = n_picks;
    p.start_with_pick = start_with_pick ? 1 : 0;
    p.tok0 = tok0;
    p.wg_picks = s.row_picks_only ? 0 : 1;
    p.epoch = s.epoch;
    p.arrive_base = s.arrive_total;
    p.spin_limit = 1u << 18;
    p.prof = s.prof;
    p.prof_cap = s.prof_cap;
    p.stop_token = -1;
    if (feed) {
        p.feed = s.feed;
        p.feed_base = s.feed_base;
        p.stop_request = s.stop_word;
        p.stop_token = stop_token;
        s.feed_base += static_cast<unsigned>(n_picks) + 1u;
    }
    PickParams& k = p.pick;
    k.logits = s.logits;
    k.V = sh.vocab;
    k.hist = s.hist;
    k.hist_stride = s.hist_stride;
    k.n_hist = s.n_hist + n_prompt;
    k.pick_idx = s.picks;
    k.tok = s.tok;
    if (o) {
        k.temperature = o->temperature;
        k.top_k = o->top_k;
        k.top_p = o->top_p;
        k.penalty = o->repetition_penalty;
        k.greedy = o->greedy;
    }
    k.uniforms = dev_uniforms;
    k.u_stride = u_stride;
    k.seed_lo = static_cast<unsigned>(seed & 0xFFFFFFFFu);
    k.seed_hi = static_cast<unsigned>(seed >> 32);
    k.work = s.work;
    k.work_stride = s.work_stride;
    k.sort_cap = kPickWorkFloats;

    if (s.xcd) {
        XcdParams x{};
        x.b = p;
        x.gm = m.xcd_geom;
        x.stream = m.xcd_stream;
        x.xc = s.xcells;
        x.ring_units = s.xcd_ring_units;
        x.ring_units_wg0 = s.xcd_ring_units_wg0;
        x.launch_base = s.xcd_launches * kWgPerXcd;
        // Eight slices per head keep the merge short; contexts beyond 256 positions give
        // every workgroup of the XCD a slice.
        x.attn_slices = (s.xcd_all_slices || s.pos + n_steps > 256) ? 0 : 8;
        s.xcd_launches++;
        hipLaunchKernelGGL(xcd_kernel_for(sh, s.xcd_row_lds, feed), dim3(kXcds * kWgPerXcd), dim3(kXcdThreads),
                           s.xcd_lds, s.stream, x);
    } else {
        PersistKernel kernel = persist_kernel_for(sh, s.pick_row_in_lds, feed);
        hipLaunchKernelGGL(kernel, dim3(s.persist_grid), dim3(kPersistThreads), s.persist_lds, s.stream, p);
    }
    HIP_CHECK(hipGetLastError());

    // Host mirrors.  Logits are produced by the last prompt step and every later one.
    int logits_phases = 0;
    for (int i = 0; i < n_steps; i++)
        if (i >= n_prompt - 1 || logit_log || i == n_steps - 1) logits_phases++;
    s.arrive_total += static_cast<unsigned>(logits_phases);
    s.epoch += static_cast<unsigned>(n_steps) + 1u;
    s.pos += n_steps;
    s.n_hist += n_prompt + n_picks;
    s.picks += n_picks;
}

// After a synchronisation of what deliver() enqueued: did the kernel give up waiting somewhere?
static void check_persist_abort(Session& s) {
    if (s.engine != GH_ENGINE_PERSISTENT) return;
    if (*s.host_err) {
        unsigned where = 0;
        HIP_CHECK(hipMemcpy(s.host_err, &s.ctl->where, sizeof(int), hipMemcpyDeviceToHost));
        where = static_cast<unsigned>(*s.host_err);
        throw ApiError{GH_ERR_DEVICE, "persistent decode kernel abandoned a wait (phase tag "
                                          + std::to_string(where) + "); the session is unusable"};
    }
}

// Makes the graph of a step's launches; returns their number.
static int record_step(Session& s, StepForm form, hipGraph_t* graph) {
    struct Scope {  // launches go to their streams again, and an unfinished graph goes, on every path out
        StepRecording recording;
        Scope() {
            HIP_CHECK(hipGraphCreate(&recording.graph, 0));
            t_recording = &recording;
        }
        ~Scope() {
            t_recording = nullptr;
            if (recording.graph) (void)hipGraphDestroy(recording.graph);
        }
    } scope;
    const int launches = enqueue_step(s, form);
    HIP_CHECK(scope.recording.error);
    *graph = scope.recording.graph;
    scope.recording.graph = nullptr;
    return launches;
}

static void run_step(Session& s, StepForm form = STEP_EMBED) {
    if (resident_now(s)) {
        enqueue_step(s, form, /*resident=*/true);
        // (embedding, layers, logits; a LayerNorm in front of the logits is a launch of its own)
        s.launches_per_step = s.m->shape.modern() ? 3 : 4;
        resident_pace(s);
        s.pos++;
        return;
    }
    s.ahead = Session::AHEAD_STREAM;
    if (s.engine == GH_ENGINE_GRAPH) {
        if (!s.exec[form]) {  // (a form's graph is made when it is first wanted)
            if (!s.graph[form]) s.form_launches[form] = record_step(s, form, &s.graph[form]);
            HIP_CHECK(hipGraphInstantiate(&s.exec[form], s.graph[form], nullptr, nullptr, 0));
        }
        s.launches_per_step = s.form_launches[form];
        HIP_CHECK(hipGraphLaunch(s.exec[form], s.stream));
    } else {
        enqueue_step(s, form);
    }
    s.pos++;
}

static void check_capacity(const Session& s) {
    // inference.cpp:151-153
    if (s.pos >= s.m->shape.max_len)
        throw ApiError{GH_ERR_RUNTIME, "InferenceSession: context exceeds max_len"};
}

static void check_ids(const Session& s, const int32_t* ids, size_t n) {
    // inference.cpp:154-156
    for (size_t i = 0; i < n; i++)
        if (ids[i] < 0 || ids[i] >= s.m->shape.vocab)
            throw ApiError{GH_ERR_OUT_OF_RANGE, "InferenceSession: token id out of vocab range"};
}

__global__ void set_state_kernel(DevState* st, int pos, int n_hist, int picks) {
    st->pos = pos;
    st->n_hist = n_hist;
    st->picks = picks;
    st->hist_lead = n_hist - pos;
}

// tok[b] = hist[b][t]
__global__ void load_tok_kernel(const int* hist, int stride, int t, int* tok, int B) {
    const int b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b < B) tok[b] = hist[static_cast<size_t>(b) * stride + t];
}

// Ids the host left in pinned memory, [B][n] on end, to rows of a device array and, of n == 1, to
// tok.  (One launch: a copy per sequence took 5 us each.)
__global__ void stage_ids_kernel(const int* __restrict__ host, size_t total, int n, int* rows, int stride, int at,
                                 int* tok) {
    const size_t i = blockIdx.x * static_cast<size_t>(blockDim.x) + threadIdx.x;
    if (i >= total) return;
    const size_t b = i / n;
    rows[b * stride + at + (i - b * n)] = host[i];
    if (tok) tok[b] = host[i];
}

static void stage_ids(Session& s, const int* host, int n, int* rows, int stride, int at, int* tok = nullptr) {
    const size_t total = static_cast<size_t>(s.B) * n;
    hipLaunchKernelGGL(stage_ids_kernel, dim3(static_cast<unsigned>((total + 255) / 256)), dim3(256), 0, s.stream, host,
                       total, n, rows, stride, at, tok);
    HIP_CHECK(hipGetLastError());
}

// What a call hands back, from device memory to pinned host memory, and with it the one-launch
// engine's error word: total 4-byte words in rows of n, which are src_stride apart there and
// follow each other here.  (One launch behind the last: each copy enqueued on its own costs 5 us
// more, a word read back by a blocking copy another 10.)
__global__ void deliver_kernel(const unsigned* __restrict__ src, size_t total, size_t n, size_t src_stride,
                               unsigned* __restrict__ dst, const unsigned* abort, int* err) {
    const size_t first = blockIdx.x * static_cast<size_t>(blockDim.x) + threadIdx.x;
    for (size_t i = first; i < total; i += gridDim.x * static_cast<size_t>(blockDim.x)) {
        const size_t b = i / n;
        dst[i] = src[b * src_stride + (i - b * n)];
    }
    if (abort && first == 0) *err = static_cast<int>(*abort);
}

// ... after which check_persist_abort needs no copy of its own.
static void deliver(Session& s, const void* src, size_t src_stride, size_t rows, size_t n, void* dst) {
    const unsigned* abort = s.engine == GH_ENGINE_PERSISTENT ? &s.ctl->abort : s.resident ? &s.rctl->abort : nullptr;
    const size_t groups = std::min<size_t>(256, std::max<size_t>(1, (rows * n + 255) / 256));
    hipLaunchKernelGGL(deliver_kernel, dim3(static_cast<unsigned>(groups)), dim3(256), 0, s.stream,
                       static_cast<const unsigned*>(src), rows * n, n, src_stride, static_cast<unsigned*>(dst), abort,
                       s.host_err);
    HIP_CHECK(hipGetLastError());
}

static void deliver_logits(Session& s) {
    const size_t V = s.m->shape.vocab;
    deliver(s, s.logits, 0, 1, s.B * V, s.host_logits);
}

// After a synchronisation of what deliver() enqueued: did a resident step give up its wait (something else held a part of
// the GPU for long)? Then the session's next steps are launches, and twice as many the next time.  A wait is
// given up after 2^18 looks, some tenths of a second: as much as the first rest, 4096 steps, loses, and a few percent of
// the longest if something is always in the way.
static bool resident_gave_up(Session& s) {
    if (!s.resident || *s.host_err == 0) return false;
    *s.host_err = 0;
    resident_end(s);
    HIP_CHECK(hipMemsetAsync(s.rctl, 0, sizeof(ResidentCtl), s.stream));  // (no step in flight, none recorded)
    s.resident_rest = s.resident_backoff;
    s.resident_backoff = std::min(2 * s.resident_backoff, 1 << 16);
    return true;
}

// Launches of a session whose steps may be resident, up to and with a deliver() and the synchronisation behind it. If a
// resident step gave up its wait, the call runs once more, as launches, from where the session stood: the
// cache rows below that position, the history and the call's ids are as they were, and what comes after is written again.
template <class Work>
static void run_resident(Session& s, Work work) {
    const int pos = s.pos, n_hist = s.n_hist, picks = s.picks;
    work();
    if (!resident_gave_up(s)) return;
    s.resident_off = true;  // until the call ends
    s.pos = pos;
    s.n_hist = n_hist;
    s.picks = picks;
    hipLaunchKernelGGL(set_state_kernel, dim3(1), dim3(1), 0, s.stream, s.st, pos, n_hist, picks);
    HIP_CHECK(hipGetLastError());
    work();
}

static void reset_session(Session& s) {
    s.pos = 0;
    s.n_hist = 0;
    s.picks = 0;
    // (the one-launch engine gets its position with the launch, and a prompt pass sets what it
    // needs of the device's copy itself)
    if (s.engine == GH_ENGINE_PERSISTENT) return;
    hipLaunchKernelGGL(set_state_kernel, dim3(1), dim3(1), 0, s.stream, s.st, 0, 0, 0);
    HIP_CHECK(hipGetLastError());
}

static std::unique_ptr<Session> create_session(const Model& m, const gh_session_opts& o) {
    require_gpu();
    if (o.batch < 1) throw ApiError{GH_ERR_INVALID_ARGUMENT, "batch must be at least 1"};
    auto sp = std::make_unique<Session>();
    Session& s = *sp;
    s.m = &m;
    s.B = o.batch;
    s.engine = o.engine;
    if (s.engine < GH_ENGINE_AUTO || s.engine > GH_ENGINE_PERSISTENT)
        throw ApiError{GH_ERR_INVALID_ARGUMENT, "unknown engine"};
    const Shape& sh = m.shape;
    int page_tokens = o.page_tokens > 0 ? o.page_tokens : 64;
    if (page_tokens & (page_tokens - 1))
        throw ApiError{GH_ERR_INVALID_ARGUMENT, "page_tokens must be a power of two"};
    // The persistent engine's offsets inside a layer's pages are 32 bits: at most 64 Ki positions in a
    // page (its contexts, 4096 at most, are one such page; longer ones of other engines take more of them).
    page_tokens = std::min(page_tokens, 1 << 16);
    s.page_shift = 0;
    while ((1 << s.page_shift) < page_tokens) s.page_shift++;
    s.pages_per_seq = (sh.max_len + page_tokens - 1) / page_tokens;
    s.n_pages = s.pages_per_seq * s.B;

    const size_t d = sh.d_model, F = sh.d_ff(), V = sh.vocab, B = s.B;
    HIP_CHECK(hipStreamCreate(&s.stream));
    for (hipEvent_t& e : s.ev) HIP_CHECK(hipEventCreate(&e));

    // Page table: identity, or a fixed scramble to exercise the indirection.
    std::vector<int> table(static_cast<size_t>(s.n_pages));
    std::iota(table.begin(), table.end(), 0);
    if (o.shuffle_pages) {
        uint64_t x = 0x9E3779B97F4A7C15ull;
        for (size_t i = table.size(); i > 1; i--) {
            x ^= x << 13;
            x ^= x >> 7;
            x ^= x << 17;
            std::swap(table[i - 1], table[x % i]);
        }
    }
    Block parts;
    parts.add(s.page_table, table.size());
    const size_t page_floats = 2ull * sh.heads * page_tokens * sh.head_size();
    parts.add(s.kv_pool, static_cast<size_t>(sh.layers) * s.n_pages * page_floats);

    parts.add(s.x, B * d);
    parts.add(s.h, B * std::max(d, F));
    parts.add(s.q, B * d);
    parts.add(s.attn, B * d);
    parts.add(s.hidden, B * F);
    parts.add(s.logits, B * V);
    s.work_stride = static_cast<int>((V + kPickThreads + 3) / 4 * 4);
    parts.add(s.work, B * static_cast<size_t>(s.work_stride));
    parts.add(s.tok, B);
    s.hist_stride = sh.max_len + 2;
    parts.add(s.hist, B * s.hist_stride);
    parts.add(s.st, 1);
    // Attention chunking: a (sequence, head) is split over several workgroups in
    // runs of 512 cache positions, or 256 when that leaves fewer than ~192
    // workgroups at a full context.  Longer runs win even when they leave compute
    // units idle (measured at context 2048 with 2..16 sequences and at context 256
    // with 8..64: every workgroup pays a dependent chain position -> page table ->
    // cache rows -> merge, and a short run does not amortise it).
    int chunk = 512;
    if (static_cast<long>(B) * sh.heads * ((sh.max_len + chunk - 1) / chunk) < 192) chunk = 256;
    if (o.flags & GH_FLAG_SMALL_ATTENTION_CHUNKS) chunk = 16;
    s.attn_chunk = chunk;
    s.attn_max_chunks = (sh.max_len + chunk - 1) / chunk;
    parts.add(s.attn_part, B * sh.heads * s.attn_max_chunks * (sh.head_size() + 2));
    parts.add(s.attn_tickets, B * sh.heads);

    // The pick keeps its working row in LDS when vocab floats fit there beside the
    // work area and the kernel's static arrays; otherwise the row stays in global
    // memory.
    int dev = 0, lds_bytes = 0;
    HIP_CHECK(hipGetDevice(&dev));
    HIP_CHECK(hipDeviceGetAttribute(&lds_bytes, hipDeviceAttributeMaxSharedMemoryPerBlock, dev));
    const size_t reserve = 8192;
    s.pick_global_scratch = (o.flags & GH_FLAG_PICK_GLOBAL_SCRATCH) != 0;
    s.row_picks_only = (o.flags & GH_FLAG_ROW_PICKS) != 0;
    s.use_prompt_pass = (o.flags & GH_FLAG_STEPWISE_PROMPT) == 0;
    s.pick_row_in_lds = !s.pick_global_scratch
                        && (V + kPickWorkFloats) * sizeof(float) + reserve <= static_cast<size_t>(lds_bytes);
    if (s.pick_row_in_lds) {
        HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(pick_kernel<true>),
                                      hipFuncAttributeMaxDynamicSharedMemorySize,
                                      lds_bytes - static_cast<int>(reserve)));
    }

    {
        int cus = 0;
        HIP_CHECK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
        const char* why = persist_unavailable(s, lds_bytes, cus);
        if (s.engine == GH_ENGINE_PERSISTENT && why) throw ApiError{GH_ERR_INVALID_ARGUMENT, why};
        if (s.engine == GH_ENGINE_AUTO) s.engine = why ? GH_ENGINE_GRAPH : GH_ENGINE_PERSISTENT;
        if (s.engine == GH_ENGINE_PERSISTENT) {
            const size_t work = d + std::max(d, F) + 192 + kPersistWaves * 4 * 68 + s.pages_per_seq;
            const size_t pick = (s.pick_row_in_lds ? V : 0) + kPickWorkFloats;
            s.persist_lds = std::max(work, pick) * sizeof(float);
            // As many workgroups as give every wavefront exactly one item of the widest phase (the
            // FFN1 row pairs): workgroups beyond that have nothing to do there and still take part
            // in every exchange.  Per token: d512 F2048 (GPT-2) 75.2 us on 256 workgroups, 67.4 on
            // 128; d768 F3072 (GPT-2) 127.0 on 256, 119.0 on 192; the Llama block d768 F2048 (2048
            // items) 116.9 on 256, 129.5 on 192.  Between these sizes every step of 16 either way
            // is slower.
            const int ffn1_items = static_cast<int>(sh.modern() ? F : F / 2);
            const int want = ((ffn1_items + kPersistWaves - 1) / kPersistWaves + 15) / 16 * 16;
            s.persist_grid = std::min(std::min(cus, 256), std::max(32, want));
            // the exchange cells, the token cell (and one of padding), then what the workgroups
            // leave for a pick each of them makes itself: nine planes of one cell per
            // workgroup and a stop word
            s.cells_count = 6 * d + F + 2 + 9 * static_cast<size_t>(s.persist_grid) + 1;
            // and, from an even index, what the workgroups that share a head's long context
            // leave for the head's own: up to fifteen shares of 66 cells for each of up to 16 heads
            s.cells_count = ((s.cells_count + 1) & ~static_cast<size_t>(1)) + 16 * 15 * 66;
            parts.add(s.cells, s.cells_count);
            parts.add(s.ctl, 1);
            if (std::getenv("GRADHIP_PROF_DUMP")) {
                s.prof_cap = 1 << 16;
                dev_alloc(s.prof, s.prof_cap);
            }
            for (const bool feed : {false, true})
                HIP_CHECK(hipFuncSetAttribute(
                    reinterpret_cast<const void*>(persist_kernel_for(sh, s.pick_row_in_lds, feed)),
                    hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(s.persist_lds)));
            s.launches_per_step = 1;

            // The XCD-sharded form, where the chip and the shape allow it: 8 XCDs of 32
            // compute units, and a ring of a power-of-two size beside the work area
            // (workgroup 0's ring is smaller when the pick keeps its row in LDS).
            XcdGeom gm;
            const bool xcd_wanted = (o.flags & GH_FLAG_XCD_PERSISTENT) != 0;
            if ((o.flags & GH_FLAG_XCD_PERSISTENT) != 0 && (o.flags & GH_FLAG_CLASSIC_PERSISTENT) != 0)
                throw ApiError{GH_ERR_INVALID_ARGUMENT, "GH_FLAG_CLASSIC_PERSISTENT and GH_FLAG_XCD_PERSISTENT exclude each other"};
            if (xcd_wanted && cus == kXcds * kWgPerXcd && xcd_geometry(sh, gm)
                && s.pages_per_seq <= 1024) {
                const size_t statics = 4096;  // the kernel's static LDS (control words, the pick's scratch), rounded up
                const size_t work = (2 * d + kWgPerXcd * kApCells + 512 + kXcdRowWaves * (128 + 32) + 192 + s.pages_per_seq)
                                    * sizeof(float);
                const size_t pick_small = kPickWorkFloats * sizeof(float);
                const size_t pick_row = (V + kPickWorkFloats) * sizeof(float);
                size_t ring = 128 * 1024;
                while (ring + std::max(work, pick_small) + statics > static_cast<size_t>(lds_bytes)) ring /= 2;
                size_t ring0 = ring;
                s.xcd_row_lds = false;
                if (!s.pick_global_scratch) {
                    size_t rr = ring;
                    while (rr >= 32 * 1024 && rr + std::max(work, pick_row) + statics > static_cast<size_t>(lds_bytes)) rr /= 2;
                    if (rr >= 32 * 1024) {
                        ring0 = rr;
                        s.xcd_row_lds = true;
                    }
                }
                if (ring >= 64 * 1024) {
                    xcd_build_stream(m);
                    s.xcd = true;
                    s.xcd_all_slices = (o.flags & GH_FLAG_SMALL_ATTENTION_CHUNKS) != 0;
                    s.xcd_ring_units = static_cast<unsigned>(ring / kXcdUnit);
                    s.xcd_ring_units_wg0 = static_cast<unsigned>(ring0 / kXcdUnit);
                    s.xcd_lds = std::max(ring + work, ring0 + std::max(work, s.xcd_row_lds ? pick_row : pick_small));
                    const XcdCells cl = xcd_cells(m.xcd_geom);
                    s.xcd_cells_count = cl.total;
                    parts.add(s.xcells, cl.total);
                    for (const bool feed : {false, true})
                        HIP_CHECK(hipFuncSetAttribute(
                            reinterpret_cast<const void*>(xcd_kernel_for(sh, s.xcd_row_lds, feed)),
                            hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(s.xcd_lds)));
                }
            }
        }
    }

    // Steps of 2 to 16 sequences: all layers in one launch, where the shape has such a kernel, it can be resident
    // (a workgroup per compute unit) and the page table fits its LDS.
    {
        int cus = 0;
        HIP_CHECK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
        const int pairs = s.B * sh.heads, runs = (sh.max_len + s.attn_chunk - 1) / s.attn_chunk;
        const size_t table_bytes = table.size() * sizeof(int);
        if (o.engine == GH_ENGINE_AUTO && s.engine == GH_ENGINE_GRAPH && resident_kernel_for(sh, s.B, pairs) && cus >= kResidentGrid
            && table_bytes <= kResidentTableBytes && s.page_shift >= 5 && s.attn_chunk % 128 == 0 && layers_back_to_back(m)) {
            s.resident = true;
            for (hipEvent_t& e : s.window_ev)  // (nobody reads memory on their word)
                HIP_CHECK(hipEventCreateWithFlags(&e, hipEventDisableTiming | hipEventDisableSystemFence));
            s.rcells_count = resident_cells(d, F, B);
            parts.add(s.rcells, s.rcells_count);
            parts.add(s.rctl, 1);
            for (int n = 1; n <= runs; n++) {  // (with the context the variant changes once)
                const ResidentKernel kernel = resident_kernel_for(sh, s.B, pairs * n);
                if (kernel && (n == 1 || kernel != resident_kernel_for(sh, s.B, pairs * (n - 1))))
                    HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                                  hipFuncAttributeMaxDynamicSharedMemorySize, kResidentTableBytes));
            }
            s.launches_per_step = sh.modern() ? 3 : 4;
            // Test aid, "looks", "looks,first" or "looks,first,launches": looks at a cell that a wait may take (0: the
            // first look has to succeed), from which of the session's resident launches on, and in how many.
            if (const char* spins = std::getenv("GRADHIP_TEST_RESIDENT_SPINS")) {
                int looks = 0, from = 0, n = INT_MAX;
                if (std::sscanf(spins, "%d,%d,%d", &looks, &from, &n) >= 1) {
                    s.spins_impatient = static_cast<unsigned>(std::min(std::max(looks, 0), 1 << 18));
                    s.impatient_from = std::max(from, 0);
                    s.impatient_n = std::max(n, 0);
                }
            }
            // ... and how many steps are launches behind the first one that gave up.
            if (const char* rest = std::getenv("GRADHIP_TEST_RESIDENT_REST"))
                s.resident_backoff = static_cast<int>(std::min(std::max(std::strtol(rest, nullptr, 10), 1l), 1l << 12));
            // ... and steps until the tags start over (as for the one-launch engine, below).
            if (const char* near = std::getenv("GRADHIP_TEST_NEAR_WRAP")) {
                const long asked = std::strtol(near, nullptr, 10);
                if (asked >= 1 && asked <= 4096)
                    s.repoch = static_cast<unsigned>(0xF0000000ull / 8ull) - static_cast<unsigned>((asked + 2) * sh.layers);
            }
        }
    }

    // The matrix-core logits launch can leave what a greedy pick needs (a batch of at
    // least two sequences takes it; the wide form and the tiled form both can).
    if (s.engine != GH_ENGINE_PERSISTENT && s.B >= kMinGemmBatch && gemm_shape_ok(sh.d_model, sh.d_model)) {
        s.best_stride = (sh.vocab + 15) / 16;
        parts.add(s.best, static_cast<size_t>(s.B) * s.best_stride);
    }

    HIP_CHECK(hipMalloc(&s.block, parts.bytes));
    parts.place(s.block);
    HIP_CHECK(hipMemsetAsync(s.block, 0, parts.bytes, s.stream));
    Block pinned;
    pinned.add(s.host_logits, B * V);
    pinned.add(s.host_ids, 2 * B * s.hist_stride);
    pinned.add(s.host_err, 1);
    pinned.add(s.feed, s.hist_stride);
    pinned.add(s.stop_word, 1);
    HIP_CHECK(hipHostMalloc(&s.host_block, pinned.bytes, hipHostMallocCoherent));
    pinned.place(s.host_block);
    std::memset(s.feed, 0, s.hist_stride * sizeof(unsigned long long));
    *s.stop_word = 0;
    *s.host_err = 0;
    HIP_CHECK(hipMemcpyAsync(s.page_table, table.data(), table.size() * sizeof(int), hipMemcpyHostToDevice, s.stream));
    if (s.engine == GH_ENGINE_PERSISTENT) {
        // Rows of the cache written earlier in a launch by other workgroups are read
        // with ordinary loads.  That is sound only because a row is never read before
        // it is written and shares no 128-byte cache line with another row: rows are
        // head_size floats from a base that hipMalloc aligns.
        if ((sh.head_size() * sizeof(float)) % 128 != 0 || reinterpret_cast<uintptr_t>(s.kv_pool) % 256 != 0)
            throw ApiError{GH_ERR_DEVICE, "persistent engine: cache rows are not whole 128-byte lines"};
        if (const char* near = std::getenv("GRADHIP_TEST_NEAR_WRAP")) {
            // Test aid: start the session's two running counts `near` steps before the
            // points where the arrival counters wrap around 2^32 and where the cell tags
            // are re-based, so that a short run crosses both.
            // (a test hook: values outside 1..4096 are ignored, so a stray variable cannot
            // leave the counters inconsistent)
            const long asked = std::strtol(near, nullptr, 10);
            const unsigned n = asked >= 1 && asked <= 4096 ? static_cast<unsigned>(asked) : 0u;
            if (n != 0u) {
                s.arrive_total = (0u - n * static_cast<unsigned>(s.persist_grid)) / static_cast<unsigned>(s.persist_grid);
                const unsigned sum = s.arrive_total * static_cast<unsigned>(s.persist_grid);
                HIP_CHECK(hipMemcpy(&s.ctl->arrive[0], &sum, sizeof(sum), hipMemcpyHostToDevice));
                s.epoch = static_cast<unsigned>(0xF0000000ull / (static_cast<unsigned long long>(sh.layers + 1) * 8ull)) - n;
            }
        }
    }
    reset_session(s);
    HIP_CHECK(hipStreamSynchronize(s.stream));

    if (s.engine == GH_ENGINE_PERSISTENT) {
        // nothing to record: one launch runs any number of steps
    } else if (!s.resident) {
        // Counts the launches of a step without running one.
        s.launches_per_step = s.form_launches[STEP_EMBED] = record_step(s, STEP_EMBED, &s.graph[STEP_EMBED]);
    }
    return sp;
}

// commit: the pick becomes part of the token history right away (the generate
// loop steps it next); otherwise the caller's following step() records it.
static void launch_pick(Session& s, const gh_sampling& o, const float* dev_uniforms, int u_stride,
                        uint64_t seed, bool commit, bool embed = false) {
    const Model& m = *s.m;
    const PickEmbed e{m.E, m.P, embed ? s.x : nullptr, m.shape.d_model, s.pos};
    PickParams p{};
    p.logits = s.logits;
    p.work = s.work;
    p.V = s.m->shape.vocab;
    p.hist = s.hist;
    p.hist_stride = s.hist_stride;
    p.n_hist = s.n_hist;
    p.pick_idx = s.picks;
    p.tok = s.tok;
    p.temperature = o.temperature;
    p.top_k = o.top_k;
    p.top_p = o.top_p;
    p.penalty = o.repetition_penalty;
    p.greedy = o.greedy;
    p.uniforms = dev_uniforms;
    p.u_stride = u_stride;
    p.seed_lo = static_cast<unsigned>(seed & 0xFFFFFFFFu);
    p.seed_hi = static_cast<unsigned>(seed >> 32);
    p.work_stride = s.work_stride;
    p.sort_cap = kPickWorkFloats;
    if (s.pick_row_in_lds) {
        hipLaunchKernelGGL(pick_kernel<true>, dim3(s.B), dim3(kPickThreads),
                           static_cast<size_t>(p.V + kPickWorkFloats) * sizeof(float), s.stream, p, e);
    } else {
        hipLaunchKernelGGL(pick_kernel<false>, dim3(s.B), dim3(kPickThreads), kPickWorkFloats * sizeof(float),
                           s.stream, p, e);
    }
    HIP_CHECK(hipGetLastError());
    if (commit) s.n_hist++;
    s.picks++;
}

static void check_sampling(const gh_sampling& o) {
    if (!o.greedy && !(o.temperature > 0.0f))
        throw ApiError{GH_ERR_INVALID_ARGUMENT, "temperature must be positive"};
    if (!(o.repetition_penalty > 0.0f))
        throw ApiError{GH_ERR_INVALID_ARGUMENT, "repetition_penalty must be positive"};
}

// ---- prompt pass: every prompt token of every sequence through each layer at once

constexpr int kPromptPassMin = 8;         // shorter prompts go token by token
constexpr size_t kPromptPassRows = 32768; // rows per pass; longer prompts run in slices

static bool prompt_pass_ok(const Session& s, int len) {
    const Shape& sh = s.m->shape;
    return s.use_prompt_pass && len >= kPromptPassMin && rows_shape_ok(sh);
}

// Passes of this many rows and more take the split projections (kernels_split.h); below,
// the small fp32 tiles of the decode step, whose norms ride inside the projections.  Speed
// alone puts the line at 160 rows (one sequence of the 69M Llama block: 128 tokens 627 us
// against 654, 244 tokens 820 against 664), and for scoring it lies there.  A prompt that is
// continued stays on the fp32 sums up to 512 rows: an unfiltered draw over a flat distribution
// of 16000 tokens falls within an fp32 rounding of the next token's boundary about once in a
// hundred picks, so the order of a prompt's sums shows in the reply, and under 512 rows the
// prompt is the small part of the request (397 tokens and 64 sampled ones: 1.4 of 12.5 ms).
// What that keeps is the replies, not precision: the split sums are the closer ones to float64.
constexpr int kSplitMinRows = 512, kSplitMinScoreRows = 160;

// How a pass over len tokens of every sequence runs: in slices of `slice` tokens (0: token by
// token), those of split_rows rows and more on the split weights.
struct RowsPlan {
    int slice = 0;
    int split_rows = 0;
    SplitKind kind = SPLIT_NONE;    // ... of those
    SplitKind logits = SPLIT_NONE;  // scored
};

// Decided before anything is launched.  Weights without a split form, or no memory for it, leave the small fp32 tiles,
// in slices below the rows from which the split projections take over (the tiles' buffers hold no
// more), and for scoring, whose logits come from the split matrix alone, the token-by-token way.
static RowsPlan plan_rows(const Session& s, int len, bool score) {
    if (!prompt_pass_ok(s, len)) return {};
    const int most = static_cast<int>(std::max<size_t>(1, std::min<size_t>(len, kPromptPassRows / s.B)));
    const long rows = static_cast<long>(most) * s.B;
    const SplitKind logits = score ? logits_kind(*s.m, rows) : SPLIT_NONE;
    if (score && logits == SPLIT_NONE) return {};
    const int split_rows = score ? kSplitMinScoreRows : kSplitMinRows;
    if (rows < split_rows) return {most, split_rows, SPLIT_NONE, logits};
    const SplitKind kind = layers_kind(*s.m, rows);
    if (kind != SPLIT_NONE) return {most, split_rows, kind, logits};
    return {std::min(len, (kSplitMinRows - 1) / s.B), kSplitMinRows, SPLIT_NONE, logits};
}

// One projection over M rows (norm folded in for RMSNorm, a norm kernel for LayerNorm).
template <int PRO, int EPI>
static void project_rows(Session& s, GemvParams g, int M) {
    hipStream_t st = s.stream;
    if (PRO == PRO_RMSNORM) {
        launch_gemm16<EPI, true>(g, M, st);
    } else {
        if (PRO == PRO_LAYERNORM) {
            launch_layernorm_rows(g.in, g.gamma, g.beta, s.pp_norm, M, g.K, st);
            HIP_CHECK(hipGetLastError());
            g.in = s.pp_norm;
            g.in_stride = g.K;
        }
        launch_gemm16<EPI, false>(g, M, st);
    }
    HIP_CHECK(hipGetLastError());
}

// Where a scored pass leaves its result: targets and nll are device arrays
// [batch][len] indexed like the ids of the pass.
struct ScoreSink {
    const int* targets;
    float* nll;
};

static SplitGemmParams split_params(const char* A, const char* W, int M, int N, int K) {
    SplitGemmParams g{};
    g.A = A;
    g.W = W;
    g.M = M;
    g.N = N;
    g.K = K;
    return g;
}

// What a product of pairs needs beside its operands: the units of W's outputs and of A.
static void pair_params(SplitGemmParams& g, const float* unit, int operand) {
    g.unit = unit;
    g.operand_unit = std::ldexp(1.0f, -operand);
}

template <int EPI>
static void split_project(Session& s, bool pairs, SplitGemmParams& g) {
    if (pairs) pair_gemm<EPI>(g, s.stream);
    else split_gemm<EPI>(g, s.stream);
}

// norm(pp_x) as an operand.
static void split_norm(Session& s, bool pairs, const float* gamma, const float* beta, int operand, int M) {
    const Shape& sh = s.m->shape;
    if (pairs)
        norm_pair(sh.modern(), s.pp_x, gamma, beta, s.pp_split, M, sh.d_model, std::ldexp(1.0f, operand), s.stream);
    else norm_split(sh.modern(), s.pp_x, gamma, beta, s.pp_split, M, sh.d_model, s.stream);
}

// Final norm, logits and the target's negative log-likelihood for rows
// pp_x[0 .. M) of a slice (row m = seq * n + t, position t0 + t).  The logits are not
// stored: every run of outputs leaves its maximum and its sum of exponentials.
static void score_rows(Session& s, const ScoreSink& sink, bool pairs, int M, int n, int t0, int len) {
    const Model& m = *s.m;
    const Shape& sh = m.shape;
    split_norm(s, pairs, m.gf, m.bf, m.logits_norm, M);
    SplitGemmParams g = split_params(s.pp_split, (pairs ? m.logits_pairs : m.logits_split).blob.at, M, sh.vocab, sh.d_model);
    if (pairs) pair_params(g, m.logits_unit, m.logits_norm);
    g.rows_per_seq = n;
    g.targets = sink.targets;
    g.nll_t0 = t0;
    g.nll_len = len;
    g.nll_part = s.nll_part;
    g.nll_target = s.nll_target;
    split_project<EPI_STORE>(s, pairs, g);
    nll_parts(g, sink.nll, s.stream);
}

static PrefillAttnParams prompt_attn_params(const Session& s, int layer, int n, int pos_base) {
    const Shape& sh = s.m->shape;
    PrefillAttnParams a{};
    a.q = s.pp_q;
    a.kv = kv_layout(s);
    a.layer = layer;
    a.d_model = sh.d_model;
    a.len = n;
    a.pos_base = pos_base;
    a.scale = 1.0f / std::sqrt(static_cast<float>(sh.head_size()));
    return a;
}

// Up to this many new tokens per sequence the fp32 kernel does a split pass's attention as
// well: splitting a context's keys and values costs as much as so few queries read of them
// (64 sequences of 128 tokens 48 us against 56, 13 of 77 10 against 18; 8 of 256 36 against 27).
// The line was drawn at position 0, where splitting weighs most: behind a cache both forms read
// what is cached, and what the split one saves grows with it.  Per layer of 12 heads, fp32 less
// split (us), 129 to 384 tokens of 1 to 32 sequences: -9..19 at position 0, 2..43 behind 256
// tokens, 50..147 behind 1024, 177..342 behind 3000.  Below the line 1 to 8 sequences would gain too
// behind a long cache (39..60 behind 1024, 160..216 behind 3000); 32 sequences would lose (5..66,
// 10..133).
// Precision, split form (2^x of scores in units of ln 2) against the fp32 one (expf), 130 to 511
// tokens at width 256, error of the losses over their size against float64: 6.7e-8..7.1e-8
// against 7.3e-8..7.9e-8 without rotation, 2.3e-7..6.5e-7 against 2.3e-7..6.6e-7 with.
constexpr int kSplitAttnMin = 128;

// The fp32 attention in blocks of 16 or of 64 queries, the same sums in either.  While the 16-query blocks
// do not fill the chip three times over what counts is the chain through a block's keys, four times as
// long with 64 queries on four wavefronts (12 heads; us per layer, 64 / 16 queries: 1 x 61 tokens 6.9 /
// 3.9, 1 x 397 31.5 / 17.6, 13 x 77 15.2 / 9.6, 3 x 333 31.5 / 19.4, 8 x 61 behind 500 48 / 27); beyond, keys read
// once for 64 queries (64 x 64 17.2 / 22.1, 64 x 128 46.8 / 65.3), unless most of a 64-query block would be
// empty (64 x 31 13.3 / 11.2, 64 x 8 behind 900 180 / 67).
template <int ROWS>
static void launch_prompt_attn_as(const Session& s, const PrefillAttnParams& a) {
    const long pairs = static_cast<long>(s.m->shape.heads) * s.B;
    const long wide = (a.len + 63) / 64 * pairs, narrow = (a.len + 15) / 16 * pairs;
    if (s.page_shift >= 6 && (narrow <= 800 || narrow <= 2 * wide))
        hipLaunchKernelGGL(attn_prefill16_kernel<ROWS>, dim3((a.len + 15) / 16, s.m->shape.heads, s.B), dim3(256), 0, s.stream, a);
    else
        hipLaunchKernelGGL(attn_prefill64_kernel<ROWS>, dim3((a.len + 63) / 64, s.m->shape.heads, s.B), dim3(256), 0, s.stream, a);
    HIP_CHECK(hipGetLastError());
}

static void launch_prompt_attn(const Session& s, const PrefillAttnParams& a) {
    if (!a.out_split) launch_prompt_attn_as<ROWS_FP32>(s, a);
    else if (a.pair_scale != 0.0f) launch_prompt_attn_as<ROWS_PAIRS>(s, a);
    else launch_prompt_attn_as<ROWS_PARTS>(s, a);
}

// One layer over M = n * B rows of pp_x through the split projections, operands in pairs or in three parts, and with
// split_attn through the split attention.  keys_only: nothing but the keys and values.
static void prompt_layer_split(Session& s, int layer, int n, int pos_base, bool pairs, bool split_attn, bool keys_only) {
    const Model& m = *s.m;
    const Shape& sh = m.shape;
    const LayerWeights& w = m.layers[layer];
    const SplitLayer sw = pairs ? SplitLayer{} : m.split_layers[layer];
    const PairLayer pw = pairs ? m.pair_layers[layer] : PairLayer{};
    const int d = sh.d_model, F = sh.d_ff(), M = n * s.B;
    hipStream_t st = s.stream;

    split_norm(s, pairs, w.g1, w.be1, pw.norm1, M);
    SplitGemmParams g = split_params(s.pp_split, pairs ? pw.wqkv : sw.wqkv, M, 3 * d, d);
    pair_params(g, pw.uqkv, pw.norm1);
    if (keys_only) {
        g.W += static_cast<size_t>(d / kSplitRows) * (d / kSplitCols) * (pairs ? kPairBlockBytes : kSplitBlockBytes);
        if (pairs) g.unit += d;
        g.N = 2 * d;
        g.first = d;
    }
    g.bias = w.bqkv;
    g.out = s.pp_q;
    g.out_stride = d;
    g.kv = kv_layout(s);
    g.layer = layer;
    g.d_model = d;
    g.rope = sh.modern();
    g.rope_cos = m.rope_cos;
    g.rope_sin = m.rope_sin;
    g.rows_per_seq = n;
    g.pos_base = pos_base;
    split_project<EPI_QKV>(s, pairs, g);
    if (keys_only) return;

    PrefillAttnParams a = prompt_attn_params(s, layer, n, pos_base);
    a.out_split = s.pp_split;
    a.pair_scale = pairs ? std::ldexp(1.0f, pw.attn) : 0.0f;
    a.key_scale = std::ldexp(1.0f, pw.keys);
    if (split_attn) split_attention(a, s.B, s.pp_kv, s.pp_kv_bytes, s.pp_part, st);
    else launch_prompt_attn(s, a);

    g = split_params(s.pp_split, pairs ? pw.wo : sw.wo, M, d, d);
    pair_params(g, pw.uo, pw.attn);
    g.bias = w.bo;
    g.out = s.pp_x;
    g.out_stride = d;
    split_project<EPI_RESID>(s, pairs, g);

    split_norm(s, pairs, w.g2, w.be2, pw.norm2, M);
    g = split_params(s.pp_split, pairs ? pw.w1 : sw.w1, M, sh.modern() ? 2 * F : F, d);
    pair_params(g, pw.u1, pw.norm2);
    g.pair_scale = std::ldexp(1.0f, pw.hidden);
    g.bias = sh.modern() ? nullptr : w.b1;
    g.out_split = s.pp_split_hidden;
    g.out_kblocks = F / kSplitCols;
    if (sh.modern()) split_project<EPI_SWIGLU>(s, pairs, g);
    else split_project<EPI_GELU>(s, pairs, g);

    g = split_params(s.pp_split_hidden, pairs ? pw.w2 : sw.w2, M, d, F);
    pair_params(g, pw.u2, pw.hidden);
    g.bias = sh.modern() ? nullptr : w.b2;
    g.out = s.pp_x;
    g.out_stride = d;
    split_project<EPI_RESID>(s, pairs, g);
}

// The same layer through the decode step's small fp32 tiles (few rows).
static void prompt_layer_small(Session& s, int layer, int n, int pos_base) {
    const Model& m = *s.m;
    const Shape& sh = m.shape;
    const LayerWeights& w = m.layers[layer];
    const int d = sh.d_model, F = sh.d_ff(), M = n * s.B;
    const bool modern = sh.modern();
    GemvParams g{};
    g.kv = kv_layout(s);
    g.layer = layer;
    g.d_model = d;
    g.st = s.st;
    g.rows_per_seq = n;
    g.pos_base = pos_base;
    g.W = w.wqkv;
    g.bias = w.bqkv;
    g.N = 3 * d;
    g.K = d;
    g.in = s.pp_x;
    g.in_stride = d;
    g.gamma = w.g1;
    g.beta = w.be1;
    g.out = s.pp_q;
    g.out_stride = d;
    g.rope = modern;
    g.rope_cos = m.rope_cos;
    g.rope_sin = m.rope_sin;
    if (modern) project_rows<PRO_RMSNORM, EPI_QKV>(s, g, M);
    else project_rows<PRO_LAYERNORM, EPI_QKV>(s, g, M);

    PrefillAttnParams a = prompt_attn_params(s, layer, n, pos_base);
    a.out = s.pp_attn;
    launch_prompt_attn(s, a);

    g.W = w.wo;
    g.bias = w.bo;
    g.N = d;
    g.K = d;
    g.in = s.pp_attn;
    g.in_stride = d;
    g.out = s.pp_x;
    g.out_stride = d;
    project_rows<PRO_PLAIN, EPI_RESID>(s, g, M);

    g.in = s.pp_x;
    g.in_stride = d;
    g.gamma = w.g2;
    g.beta = w.be2;
    g.out = s.pp_hidden;
    g.out_stride = F;
    g.W = w.w1;
    g.K = d;
    if (modern) {
        g.bias = nullptr;
        g.N = 2 * F;
        project_rows<PRO_RMSNORM, EPI_SWIGLU>(s, g, M);
    } else {
        g.bias = w.b1;
        g.N = F;
        project_rows<PRO_LAYERNORM, EPI_GELU>(s, g, M);
    }
    g.W = w.w2;
    g.bias = modern ? nullptr : w.b2;
    g.N = d;
    g.K = F;
    g.in = s.pp_hidden;
    g.in_stride = F;
    g.out = s.pp_x;
    g.out_stride = d;
    project_rows<PRO_PLAIN, EPI_RESID>(s, g, M);
}

// The session's buffer p of n elements, cleared, in place of the one it had.
template <typename T>
static bool replace_buffer(Session& s, T*& p, size_t n) {
    if (p) HIP_CHECK(hipFree(p));
    if (!try_alloc(p, n)) return false;
    HIP_CHECK(hipMemsetAsync(p, 0, std::max<size_t>(n, 1) * sizeof(T), s.stream));
    return true;
}

// Activations of a prompt pass of up to `rows` rows (grown on demand).  False: not enough memory.
static bool reserve_prompt_rows(Session& s, size_t rows) {
    const size_t d = s.m->shape.d_model, F = s.m->shape.d_ff();
    if (s.pp_rows >= rows) return true;
    s.pp_rows = 0;
    const size_t few = std::min<size_t>(rows, kSplitMinRows);  // what the small tiles still take
    const bool all = replace_buffer(s, s.pp_x, rows * d) && replace_buffer(s, s.pp_q, rows * d)
                     && replace_buffer(s, s.pp_attn, few * d) && replace_buffer(s, s.pp_norm, few * d)
                     && replace_buffer(s, s.pp_hidden, few * F) && replace_buffer(s, s.pp_split, split_bytes(rows, d))
                     && replace_buffer(s, s.pp_split_hidden, split_bytes(rows, F));
    if (all) s.pp_rows = rows;
    return all;
}

// What scoring leaves of that many rows' logits.
static bool reserve_score_rows(Session& s, size_t rows) {
    if (s.nll_rows >= rows) return true;
    s.nll_rows = 0;
    const bool all = replace_buffer(s, s.nll_part, rows * split_nll_stride(s.m->shape.vocab))
                     && replace_buffer(s, s.nll_target, rows);
    if (all) s.nll_rows = rows;
    return all;
}

// Scratch of a split pass's attention over n new positions behind pos_base: for keys and values what
// the session's whole context can use, so that it is allocated once (nothing in it is read that the
// pass has not written, so it is not cleared); partial results grow in steps of 8 MB, up to some 45.
// False: there is no memory, or too little work; the fp32 kernel, which needs none, does it.
static bool reserve_split_attention(Session& s, int n, int pos_base, bool pairs) {
    if (n <= kSplitAttnMin) return false;
    const int heads = s.m->shape.heads;
    if (!s.pp_kv) {
        const size_t bytes = split_attention_kv_bytes(s.B, heads, s.m->shape.max_len);
        if (!try_alloc(s.pp_kv, bytes)) return false;
        s.pp_kv_bytes = bytes;
    }
    const size_t need = split_attention_part_floats(s.B, heads, n, pos_base, s.pp_kv_bytes, pairs);
    if (s.pp_part_floats < need) {
        if (s.pp_part) HIP_CHECK(hipFree(s.pp_part));
        s.pp_part_floats = 0;
        const size_t floats = align_up(need, size_t{2} << 20);
        if (!try_alloc(s.pp_part, floats)) return false;
        s.pp_part_floats = floats;
    }
    return true;
}

// Tokens hist[n_hist .. n_hist + len) of every sequence, positions pos .. pos + len.
// Equivalent to len step() calls (text_gen.cpp:44-46); only the last logits are
// formed unless a sink asks for the likelihood of a target at every position.
static void prompt_pass(Session& s, int len, const RowsPlan& plan, const ScoreSink* sink = nullptr) {
    const Model& m = *s.m;
    const Shape& sh = m.shape;
    const int d = sh.d_model, B = s.B;
    hipStream_t st = s.stream;
    // (too little memory for the slices: shorter ones, down to the rows that the small tiles take)
    int slice = plan.slice;
    const auto reserved = [&] {
        const size_t rows = static_cast<size_t>(slice) * B;
        return reserve_prompt_rows(s, rows) && (!sink || reserve_score_rows(s, rows));
    };
    while (!reserved()) {
        if (slice == 1 || slice * B < kSplitMinRows) throw ApiError{GH_ERR_DEVICE, "out of device memory for a prompt pass"};
        slice = (slice + 1) / 2;
    }
    // Whether the layers and the scored logits of n tokens go in pairs: a shorter slice's form is its own, the others' if there is
    // no memory for it.  Made, like the plan's, before anything is launched.
    const auto in_pairs = [&](int n) {
        const auto kind = [&](SplitKind planned, auto kind_of) {
            const SplitKind own = n == plan.slice ? planned : kind_of(m, static_cast<long>(n) * B);
            return (own == SPLIT_NONE ? planned : own) == SPLIT_PAIRS;
        };
        return std::make_pair(n * B >= plan.split_rows && kind(plan.kind, layers_kind), sink && kind(plan.logits, logits_kind));
    };
    const auto whole = in_pairs(slice), last = in_pairs((len - 1) % slice + 1);
    for (int t0 = 0; t0 < len; t0 += slice) {
        const int n = std::min(slice, len - t0);
        const int M = n * B;
        const int pos_base = s.pos + t0;
        const bool split = M >= plan.split_rows;
        const bool pairs = split && (n == slice ? whole : last).first;
        const bool split_attn = split && reserve_split_attention(s, n, pos_base, pairs);
        hipLaunchKernelGGL(embed_rows_kernel, dim3((d + 255) / 256, M), dim3(256), 0, st, m.E, m.P, s.hist,
                           s.hist_stride, s.n_hist + t0, n, pos_base, s.pp_x, d);
        HIP_CHECK(hipGetLastError());
        // Of the last layer a pass that is not scored needs the keys and values, and everything
        // else at the last position alone, where the decode step's launches are as good.
        const bool trim = split && !sink;
        for (int l = 0; l < sh.layers; l++) {
            if (split) prompt_layer_split(s, l, n, pos_base, pairs, split_attn, trim && l == sh.layers - 1);
            else prompt_layer_small(s, l, n, pos_base);
        }
        if (sink) score_rows(s, *sink, (n == slice ? whole : last).second, M, n, t0, len);
        if (t0 + n == len) {
            hipLaunchKernelGGL(take_last_rows_kernel, dim3((d + 255) / 256, B), dim3(256), 0, st, s.pp_x, n,
                               s.x, d);
            HIP_CHECK(hipGetLastError());
            if (trim) {
                hipLaunchKernelGGL(set_state_kernel, dim3(1), dim3(1), 0, st, s.st, pos_base + n - 1, s.n_hist, s.picks);
                HIP_CHECK(hipGetLastError());
                enqueue_layer(s, sh.layers - 1, /*query_only=*/true);
            }
        }
    }
    s.pos += len;
    s.n_hist += len;
    hipLaunchKernelGGL(set_state_kernel, dim3(1), dim3(1), 0, st, s.st, s.pos, s.n_hist, s.picks);
    HIP_CHECK(hipGetLastError());
    // logits of the last position, through the decode-size projection
    enqueue_logits(s, /*advance=*/false);
}

// Steps through `len` tokens already staged in the history at n_hist.. (the
// prompt loop of text_gen.cpp:44-46).  log: per-step logits destination or null.
static void run_prompt(Session& s, int len, float* log, size_t* steps_logged) {
    const size_t BV = static_cast<size_t>(s.B) * s.m->shape.vocab;
    const RowsPlan plan = log ? RowsPlan{} : plan_rows(s, len, /*score=*/false);
    if (plan.slice > 0) {
        prompt_pass(s, len, plan);
        if (steps_logged) *steps_logged += len;
        return;
    }
    if (s.engine == GH_ENGINE_PERSISTENT) {
        persist_run(s, len, len, 0, false, nullptr, nullptr, 0, 0,
                    log ? log + *steps_logged * BV : nullptr);
        if (steps_logged) *steps_logged += len;
        return;
    }
    const int base = s.n_hist;
    for (int t = 0; t < len; t++) {
        hipLaunchKernelGGL(load_tok_kernel, dim3((s.B + 63) / 64), dim3(64), 0, s.stream, s.hist,
                           s.hist_stride, base + t, s.tok, s.B);
        HIP_CHECK(hipGetLastError());
        run_step(s);
        if (log) {
            HIP_CHECK(hipMemcpyAsync(log + *steps_logged * BV, s.logits, BV * sizeof(float),
                                     hipMemcpyDeviceToDevice, s.stream));
        }
        if (steps_logged) (*steps_logged)++;
    }
    s.n_hist += len;
}

// The decode loop of text_gen.cpp:48-64 from the current context: pick, push,
// stop at capacity, else step.  Returns {picks made, steps run}.
static std::pair<int, int> run_decode(Session& s, int max_tokens, const gh_sampling& o,
                                      const float* du, int u_stride, uint64_t seed, float* log,
                                      size_t* steps_logged) {
    const int C = s.m->shape.max_len;
    const size_t BV = static_cast<size_t>(s.B) * s.m->shape.vocab;
    if (s.engine == GH_ENGINE_PERSISTENT) {
        int picks = 0, steps = 0, pos = s.pos, nh = s.n_hist;
        for (int i = 0; i < max_tokens; i++) {
            if (nh >= s.hist_stride) break;
            picks++;
            nh++;
            if (pos >= C) break;
            steps++;
            pos++;
        }
        persist_run(s, 0, steps, picks, true, &o, du, u_stride, seed,
                    log ? log + *steps_logged * BV : nullptr);
        if (steps_logged) *steps_logged += steps;
        return {picks, steps};
    }
    // Greedy without a penalty on the matrix-core path: after the first step of the call
    // the pick rides at the head of the next step (the logits launch left what it needs).
    const bool pick_rides = s.best && o.greedy && o.repetition_penalty == 1.0f;
    if (pick_rides) {
        hipLaunchKernelGGL(set_state_kernel, dim3(1), dim3(1), 0, s.stream, s.st, s.pos, s.n_hist, s.picks);
        HIP_CHECK(hipGetLastError());
    }
    int picks = 0, steps = 0;
    for (int i = 0; i < max_tokens; i++) {
        if (s.n_hist >= s.hist_stride) break;
        const bool riding = pick_rides && steps > 0 && s.pos < C;
        if (riding) {
            s.n_hist++;
            s.picks++;
        } else {
            launch_pick(s, o, du, u_stride, seed, true, /*embed=*/s.pos < C);
        }
        picks++;
        if (s.pos >= C) break;
        run_step(s, riding ? STEP_ARGMAX : STEP_ROWS);
        steps++;
        if (log) {
            HIP_CHECK(hipMemcpyAsync(log + *steps_logged * BV, s.logits, BV * sizeof(float),
                                     hipMemcpyDeviceToDevice, s.stream));
        }
        if (steps_logged) (*steps_logged)++;
    }
    return {picks, steps};
}

// The logits that a run of steps begins with, kept while its steps may be resident: the first pick is
// made from them and the steps overwrite them.  (Without memory for the copy the launches do.)
static void keep_logits(Session& s, bool restore) {
    const size_t n = static_cast<size_t>(s.B) * s.m->shape.vocab;
    if (restore) {
        HIP_CHECK(hipMemcpyAsync(s.logits, s.start_logits, n * sizeof(float), hipMemcpyDeviceToDevice, s.stream));
        return;
    }
    if (!s.resident) return;
    if (!s.start_logits && !try_alloc(s.start_logits, n)) {
        s.resident_off = true;  // for this call
        return;
    }
    HIP_CHECK(hipMemcpyAsync(s.start_logits, s.logits, n * sizeof(float), hipMemcpyDeviceToDevice, s.stream));
}

// In a streamed run, after a synchronisation: if the last step was resident and gave up, it runs again as launches.
// picked: a pick made from its logits is to be forgotten.  True if it had to.
static bool repeat_step(Session& s, bool picked) {
    if (!resident_gave_up(s)) return false;
    s.pos--;
    if (picked) {
        s.n_hist--;
        s.picks--;
    }
    hipLaunchKernelGGL(set_state_kernel, dim3(1), dim3(1), 0, s.stream, s.st, s.pos, s.n_hist, s.picks);
    hipLaunchKernelGGL(load_tok_kernel, dim3((s.B + 63) / 64), dim3(64), 0, s.stream, s.hist, s.hist_stride, s.n_hist - 1, s.tok,
                       s.B);
    HIP_CHECK(hipGetLastError());
    run_step(s);
    return true;
}

// Copies the caller's uniforms to the device (grown on demand); null for none.
static const float* stage_uniforms(Session& s, const float* uniforms, size_t n) {
    if (!uniforms || n == 0) return nullptr;
    if (s.uniforms_cap < n) {
        if (s.uniforms) HIP_CHECK(hipFree(s.uniforms));
        s.uniforms = nullptr;
        dev_alloc(s.uniforms, n);
        s.uniforms_cap = n;
    }
    HIP_CHECK(hipMemcpyAsync(s.uniforms, uniforms, n * sizeof(float), hipMemcpyHostToDevice, s.stream));
    return s.uniforms;
}

// ---- a pick that allocates nothing (gh_pick_noalloc)

// The sampler's working rows for callers that cannot allocate: one array per
// GPU, held until the process ends.  Host code never uses this name as an
// address; it asks the runtime where the array lives on the current device.
constexpr size_t kNoAllocScratchFloats = size_t{1} << 20;  // 4 MiB
static __device__ __align__(256) float scratch[kNoAllocScratchFloats];

__global__ __launch_bounds__(kPickThreads) void pick_noalloc_kernel(const PickParams p, int* out_ids) {
    extern __shared__ __attribute__((aligned(128))) float lds[];
    const int b = blockIdx.x;
    const int chosen = pick_body<false, kPickThreads, false>(p, b, p.work + static_cast<size_t>(b) * p.work_stride, lds);
    if (threadIdx.x == 0) out_ids[b] = chosen;
}

constexpr int kMaxDevices = 64;
static std::mutex g_scratch_mutex;
static float* g_scratch_ptr[kMaxDevices] = {};

// Device address of `scratch` on the current GPU, looked up once per device.
static float* scratch_on_current_device() {
    int dev = 0;
    HIP_CHECK(hipGetDevice(&dev));
    if (dev < 0 || dev >= kMaxDevices) throw ApiError{GH_ERR_DEVICE, "device index beyond the scratch table"};
    std::lock_guard<std::mutex> lk(g_scratch_mutex);
    if (!g_scratch_ptr[dev]) {
        float* ptr = nullptr;
        HIP_CHECK(hipGetSymbolAddress(reinterpret_cast<void**>(&ptr), HIP_SYMBOL(scratch)));
        if (!ptr) throw ApiError{GH_ERR_DEVICE, "the scratch array has no address on this device"};
        g_scratch_ptr[dev] = ptr;
    }
    return g_scratch_ptr[dev];
}

// ---- matrix-core issue probe (gh_device_mfma_issue)

// Wavefronts 0-3 of a workgroup (one per SIMD) run a dependent chain of fp32 matrix
// products, wavefronts 4-7 (the same SIMDs) runs of VPER dependent-free multiply-adds,
// or wavefronts 0-3 both in turn; every wavefront reports its shader-clock cycles.
template <int VPER>
__global__ __launch_bounds__(512) void mfma_issue_probe_kernel(long long* out, int iters, int mode, float a, float b) {
    typedef float v16f __attribute__((ext_vector_type(16)));
    const int wave = threadIdx.x >> 6;
    v16f acc;
#pragma unroll
    for (int r = 0; r < 16; r++) acc[r] = 0.0f;
    float x[8];
#pragma unroll
    for (int i = 0; i < 8; i++) x[i] = a + static_cast<float>(i);
    __syncthreads();
    const long long c0 = clock64(), w0 = wall_clock64();
    if (wave < 4) {
        if (mode & 1) {
            for (int i = 0; i < iters; i++) {
#pragma unroll
                for (int u = 0; u < 8; u++) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, acc, 0, 0, 0);
            }
        } else if (mode & 4) {
            for (int i = 0; i < iters; i++) {
#pragma unroll
                for (int u = 0; u < 8; u++) {
                    acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, acc, 0, 0, 0);
#pragma unroll
                    for (int v = 0; v < VPER; v++) x[v & 7] = x[v & 7] * b + a;
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        }
    } else if (mode & 2) {
        for (int i = 0; i < iters; i++) {
#pragma unroll
            for (int u = 0; u < 8; u++) {
#pragma unroll
                for (int v = 0; v < VPER; v++) x[v & 7] = x[v & 7] * b + a;
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    }
    const long long c1 = clock64(), w1 = wall_clock64();
    float keep = acc[0];
#pragma unroll
    for (int i = 0; i < 8; i++) keep += x[i];
    if ((threadIdx.x & 63) == 0) {
        long long* o = out + (static_cast<size_t>(blockIdx.x) * 8 + wave) * 3;
        o[0] = c1 - c0;
        o[1] = w1 - w0;
        o[2] = static_cast<long long>(keep);
    }
}

// ---- hand-off latency probe (gh_device_handoff_latency)

// Workgroup 0 and workgroup `peer` bounce a counter: each waits until the other's word
// has reached the round number and then writes its own.  LOAD: cache policy of the
// polling load (buffer aux bits); DEVICE_STORE: device-scope (write-through) store or
// an ordinary one.  Bounded polling: a side that never sees its peer gives up.
template <int LOAD, bool DEVICE_STORE>
__global__ void handoff_probe_kernel(unsigned* cells, int peer, int rounds, unsigned long long* ticks, unsigned* xcds) {
    const int me = blockIdx.x == 0 ? 0 : (static_cast<int>(blockIdx.x) == peer ? 1 : -1);
    if (threadIdx.x == 0) xcds[blockIdx.x] = xcc_id();
    if (me < 0 || threadIdx.x != 0) return;
    unsigned* mine = cells + me * 64;
    const __amdgpu_buffer_rsrc_t rs = make_buffer(cells + (1 - me) * 64, 4);
    auto put = [&](unsigned v) {
        if (DEVICE_STORE) __hip_atomic_store(mine, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        else *reinterpret_cast<volatile unsigned*>(mine) = v;
    };
    const unsigned long long t0 = __builtin_amdgcn_s_memrealtime();
    for (int i = 1; i <= rounds; i++) {
        if (me == 0) put(static_cast<unsigned>(i));
        unsigned spins = 0;
        while (static_cast<unsigned>(__builtin_amdgcn_raw_buffer_load_b32(rs, 0, 0, LOAD)) < static_cast<unsigned>(i)
               && ++spins < (1u << 20)) {
        }
        if (me == 1) put(static_cast<unsigned>(i));
    }
    ticks[me] = __builtin_amdgcn_s_memrealtime() - t0;  // 100 MHz
}

// Background load for the probe: streams a buffer until told to stop (or 2000 rounds).
__global__ void handoff_probe_hog(const float4* buf, size_t n4, const volatile unsigned* stop, float* sink) {
    float acc = 0.0f;
    size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    const size_t stride = static_cast<size_t>(gridDim.x) * blockDim.x;
    for (int it = 0; it < 2000 && *stop == 0u; it++)
        for (int k = 0; k < 16; k++) {
            const float4 v = buf[i];
            acc += (v.x + v.y) + (v.z + v.w);
            i += stride;
            if (i >= n4) i -= n4;
        }
    if (acc == 1.2345f) *sink = acc;
}

using HandoffKernel = void (*)(unsigned*, int, int, unsigned long long*, unsigned*);
static HandoffKernel handoff_kernel_for(int load_policy, bool device_store) {
    switch (load_policy) {
    case 0: return device_store ? handoff_probe_kernel<0, true> : handoff_probe_kernel<0, false>;
    case 1: return device_store ? handoff_probe_kernel<kAuxNonTemporal, true> : handoff_probe_kernel<kAuxNonTemporal, false>;
    case 2: return device_store ? handoff_probe_kernel<kAuxDeviceScope, true> : handoff_probe_kernel<kAuxDeviceScope, false>;
    default: return nullptr;
    }
}

}  // namespace gh

// ====================================================================== C ABI

using namespace gh;

struct gh_model {
    std::unique_ptr<Model> impl;
};
struct gh_session {
    std::unique_ptr<Session> impl;
};

// A plain streaming read (eight 16-byte loads in flight per thread): what a
// bandwidth-bound kernel can reach on this device.
__global__ __launch_bounds__(256) void stream_read_kernel(const float4* __restrict__ a, size_t n4, float* sink) {
    float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
    const size_t stride = static_cast<size_t>(gridDim.x) * blockDim.x;
    size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    for (; i + 7 * stride < n4; i += 8 * stride) {
        float4 v[8];
#pragma unroll
        for (int u = 0; u < 8; u++) v[u] = a[i + u * stride];
#pragma unroll
        for (int u = 0; u < 8; u++) {
            acc.x += v[u].x;
            acc.y += v[u].y;
            acc.z += v[u].z;
            acc.w += v[u].w;
        }
    }
    for (; i < n4; i += stride) {  // what is left (all of a buffer below 256 MiB)
        const float4 v = a[i];
        acc.x += v.x;
        acc.y += v.y;
        acc.z += v.z;
        acc.w += v.w;
    }
    if (acc.x + acc.y + acc.z + acc.w == 12345.0f) *sink = 1.0f;  // keeps the loads alive
}

extern "C" {

const char* gh_last_error(void) { return g_last_error.c_str(); }

// ---- tokenizer (host only)

// Exactly one of the two is set.
struct gh_tokenizer {
    std::optional<gh::ByteBpe> v2;
    std::optional<gh::BpeV1> v1;
};

gh_status gh_tokenizer_load(const char* path, gh_tokenizer** out) {
    return guard([&] {
        if (!path || !out) throw ApiError{GH_ERR_INVALID_ARGUMENT, "null argument"};
        *out = nullptr;
        // anything that does not start with "GTOK" is taken for a v1 cache (tokenizer.cpp:107-117)
        if (is_gtok_file(path)) *out = new gh_tokenizer{ByteBpe::load(path), std::nullopt};
        else *out = new gh_tokenizer{std::nullopt, BpeV1::load(path)};
    });
}

gh_status gh_tokenizer_from_merges(const int32_t* merges, int32_t n_merges, const char* const* specials,
                                   const int32_t* special_lens, int32_t n_specials, gh_tokenizer** out) {
    return guard([&] {
        if (!out || n_merges < 0 || n_specials < 0 || (n_merges > 0 && !merges)
            || (n_specials > 0 && (!specials || !special_lens)))
            throw ApiError{GH_ERR_INVALID_ARGUMENT, "null argument"};
        *out = nullptr;
        std::vector<ByteBpe::Merge> m;
        m.reserve(static_cast<size_t>(n_merges));
        for (int32_t r = 0; r < n_merges; r++) m.emplace_back(merges[2 * r], merges[2 * r + 1]);
        std::vector<std::string> sp;
        for (int32_t i = 0; i < n_specials; i++)
            sp.emplace_back(specials[i], static_cast<size_t>(std::max(special_lens[i], 0)));
        *out = new gh_tokenizer{ByteBpe(std::move(m), std::move(sp)), std::nullopt};
    });
}

gh_status gh_tokenizer_save(const gh_tokenizer* t, const char* path) {
    return guard([&] {
        if (!t || !path) throw ApiError{GH_ERR_INVALID_ARGUMENT, "null argument"};
        if (t->v2) t->v2->save(path);
        else t->v1->save(path);
    });
}

void gh_tokenizer_free(gh_tokenizer* t) { delete t; }

gh_status gh_tokenizer_get_info(const gh_tokenizer* t, gh_tokenizer_info* out) {
    return guard([&] {
        if (!t || !out) throw ApiError{GH_ERR_INVALID_ARGUMENT, "null argument"};
        if (t->v2) {
            out->kind = ByteBpe::kKind;
            out->vocab_size = t->v2->vocab_size();
            out->eos_id = t->v2->special_id("<|endoftext|>");  // byte_bpe.h:78
            out->n_merges = static_cast<int32_t>(t->v2->merges().size());
            out->n_specials = static_cast<int32_t>(t->v2->specials().size());
            out->fingerprint = t->v2->fingerprint();
        } else {
            out->kind = BpeV1::kKind;
            out->vocab_size = t->v1->vocab_size();
            out->eos_id = t->v1->special_id("<eos>");  // tokenizer.cpp:95-97
            out->n_merges = static_cast<int32_t>(t->v1->merge_count());
            out->n_specials = 0;
            for (const char* sp : {"<pad>", "<eos>", "<unk>"}) out->n_specials += t->v1->special_id(sp) >= 0;
            out->fingerprint = t->v1->fingerprint();
        }
    });
}

gh_status gh_tokenizer_special_id(const gh_tokenizer* t, const char* token, size_t len, int32_t* id) {
    return guard([&] {
        if (!t || !id || (len > 0 && !token)) throw ApiError{GH_ERR_INVALID_ARGUMENT, "null argument"};
        const std::string_view tv(token, len);
        *id = t->v2 ? t->v2->special_id(tv) : t->v1->special_id(tv);
    });
}

gh_status gh_tokenizer_encode(const gh_tokenizer* t, const char* text, size_t len, int32_t with_specials,
                              int32_t* ids, size_t cap, size_t* n) {
    return guard([&] {
        if (!t || !n || (len > 0 && !text) || (cap > 0 && !ids))
            throw ApiError{GH_ERR_INVALID_ARGUMENT, "null argument"};
        const std::string_view tv(text, len);
        const std::vector<int> got = t->v2 ? t->v2->encode(tv, with_specials != 0) : t->v1->encode(tv);
        *n = got.size();
        std::copy_n(got.begin(), std::min(cap, got.size()), ids);
    });
}

gh_status gh_tokenizer_decode(const gh_tokenizer* t, const int32_t* ids, size_t n, char* out, size_t cap,
                              size_t* len) {
    return guard([&] {
        if (!t || !len || (n > 0 && !ids) || (cap > 0 && !out))
            throw ApiError{GH_ERR_INVALID_ARGUMENT, "null argument"};
        const std::string got = t->v2 ? t->v2->decode(ids, n) : t->v1->decode(ids, n);
        *len = got.size();
        std::copy_n(got.begin(), std::min(cap, got.size()), out);
    });
}

gh_status gh_pretokenize(const char* text, size_t len, size_t* ends, size_t cap, size_t* n) {
    return guard([&] {
        if (!n || (len > 0 && !text) || (cap > 0 && !ends)) throw ApiError{GH_ERR_INVALID_ARGUMENT, "null argument"};
        const std::string_view v(text, len);
        size_t pieces = 0;
        for (size_t pos = 0; pos < len;) {
            pos = pretok::piece_end(v, pos);
            if (pieces < cap) ends[pieces] = pos;
            pieces++;
        }
        *n = pieces;
    });
}

int32_t gh_codepoint_class(uint32_t codepoint) { return pretok::classify(codepoint); }

static Shape shape_of(const gh_config& c) {
    Shape s;
    s.arch = c.arch;
    s.vocab = c.vocab;
    s.d_model = c.d_model;
    s.layers = c.layers;
    s.heads = c.heads;
    s.max_len = c.max_len;
    s.dropout = c.dropout;
    return s;
}

static void check_config(const gh_config* cfg) {
    if (!cfg) throw ApiError{GH_ERR_INVALID_ARGUMENT, "null config"};
    if (cfg->arch != GH_ARCH_GPT2 && cfg->arch != GH_ARCH_MODERN)
        throw ApiError{GH_ERR_RUNTIME, "unknown architecture tag " + std::to_string(cfg->arch)};
    validate_shape(shape_of(*cfg));
}

gh_status gh_model_load(const char* path, gh_model** out) {
    return guard([&] {
        if (!path || !out) throw ApiError{GH_ERR_INVALID_ARGUMENT, "null argument"};
        *out = nullptr;
        HostModel hm = read_checkpoint(path);
        std::vector<const float*> ptrs;
        for (const auto& t : hm.tensors) ptrs.push_back(t.data());
        try {
            auto m = upload_model(hm.shape, ptrs, hm.tokenizer);
            *out = new gh_model{std::move(m)};
        } catch (const ApiError& e) {
            throw ApiError{e.code, std::string("Failed to load model from ") + path + ": " + e.msg};
        }
    });
}

gh_status gh_model_from_host(const gh_config* cfg, const float* const* tensors, int32_t n_tensors,
                             gh_model** out) {
    return guard([&] {
        if (!tensors || !out) throw ApiError{GH_ERR_INVALID_ARGUMENT, "null argument"};
        *out = nullptr;
        check_config(cfg);
        const Shape s = shape_of(*cfg);
        if (static_cast<size_t>(n_tensors) != tensor_specs(s).size())
            throw ApiError{GH_ERR_INVALID_ARGUMENT, "tensor count does not match the model shape"};
        std::vector<const float*> ptrs(tensors, tensors + n_tensors);
        for (const float* p : ptrs)
            if (!p) throw ApiError{GH_ERR_INVALID_ARGUMENT, "null tensor"};
        std::optional<Fingerprint> fp;
        if (cfg->has_fingerprint) fp = Fingerprint{cfg->tokenizer_kind, cfg->tokenizer_hash};
        *out = new gh_model{upload_model(s, ptrs, fp)};
    });
}

int32_t gh_config_num_tensors(const gh_config* cfg) {
    int32_t n = -1;
    (void)guard([&] {
        check_config(cfg);
        n = static_cast<int32_t>(tensor_specs(shape_of(*cfg)).size());
    });
    return n;
}

gh_status gh_config_tensor_shape(const gh_config* cfg, int32_t index, int32_t* rows, int32_t* cols) {
    return guard([&] {
        check_config(cfg);
        const auto specs = tensor_specs(shape_of(*cfg));
        if (index < 0 || static_cast<size_t>(index) >= specs.size())
            throw ApiError{GH_ERR_OUT_OF_RANGE, "tensor index out of range"};
        if (rows) *rows = specs[index].rows;
        if (cols) *cols = specs[index].cols;
    });
}

gh_status gh_model_save(const gh_model* m, const char* path) {
    return guard([&] {
        if (!m || !path) throw ApiError{GH_ERR_INVALID_ARGUMENT, "null argument"};
        const auto host = download_model(*m->impl);
        std::vector<const float*> ptrs;
        for (const auto& t : host) ptrs.push_back(t.data());
        std::string why;
        if (!write_checkpoint(path, m->impl->shape, ptrs, m->impl->tokenizer, why))
            throw ApiError{GH_ERR_RUNTIME, why};
    });
}

void gh_model_free(gh_model* m) { delete m; }

gh_status gh_model_get_config(const gh_model* m, gh_config* out) {
    return guard([&] {
        if (!m || !out) throw ApiError{GH_ERR_INVALID_ARGUMENT, "null argument"};
        const Shape& s = m->impl->shape;
        *out = gh_config{};
        out->arch = s.arch;
        out->vocab = s.vocab;
        out->d_model = s.d_model;
        out->layers = s.layers;
        out->heads = s.heads;
        out->max_len = s.max_len;
        out->d_ff = s.d_ff();
        out->dropout = s.dropout;
        if (m->impl->tokenizer) {
            out->has_fingerprint = 1;
            out->tokenizer_kind = m->impl->tokenizer->kind;
            out->tokenizer_hash = m->impl->tokenizer->hash;
        }
    });
}

gh_status gh_session_create(const gh_model* m, const gh_session_opts* opts, gh_session** out) {
    return guard([&] {
        if (!m || !out) throw ApiError{GH_ERR_INVALID_ARGUMENT, "null argument"};
        *out = nullptr;
        gh_session_opts o{};
        o.batch = 1;
        if (opts) o = *opts;
        *out = new gh_session{create_session(*m->impl, o)};
    });
}

void gh_session_free(gh_session* s) { delete s; }

gh_status gh_session_reset(gh_session* s) {
    return guard([&] {
        if (!s) throw ApiError{GH_ERR_INVALID_ARGUMENT, "null session"};
        reset_session(*s->impl);
        if (s->impl->engine != GH_ENGINE_PERSISTENT) HIP_CHECK(hipStreamSynchronize(s->impl->stream));
    });
}

gh_status gh_session_step(gh_session* sess, const int32_t* ids, float* logits_host) {
    return guard([&] {
        if (!sess || !ids) throw ApiError{GH_ERR_INVALID_ARGUMENT, "null argument"};
        Session& s = *sess->impl;
        const PersistGate gate(s);  // held until this call has synchronised its launches
        const ResidentScope scope(s);
        check_capacity(s);
        check_ids(s, ids, s.B);
        const size_t V = s.m->shape.vocab;
        const bool one_launch = s.engine == GH_ENGINE_PERSISTENT && s.n_hist == s.pos;
        if (one_launch) {
            // The token travels in the kernel's arguments (the kernel records it in the history,
            // whose index is the position).
            persist_run(s, 1, 1, 0, false, nullptr, nullptr, 0, 0, nullptr, false, -1, ids[0]);
        } else {
            std::memcpy(s.host_ids, ids, s.B * sizeof(int));
            // The history (index == position) feeds the repetition penalty of later picks.
            stage_ids(s, s.host_ids, 1, s.hist, s.hist_stride, s.n_hist, s.tok);
            if (s.engine == GH_ENGINE_PERSISTENT) persist_run(s, 1, 1, 0, false, nullptr, nullptr, 0, 0, nullptr);
        }
        run_resident(s, [&] {
            if (s.engine != GH_ENGINE_PERSISTENT) {
                s.n_hist++;
                run_step(s);
            }
            deliver_logits(s);
            HIP_CHECK(hipStreamSynchronize(s.stream));
        });
        check_persist_abort(s);
        if (logits_host) std::memcpy(logits_host, s.host_logits, s.B * V * sizeof(float));
    });
}

gh_status gh_session_logits(gh_session* s, const float** logits) {
    return guard([&] {
        if (!s || !logits) throw ApiError{GH_ERR_INVALID_ARGUMENT, "null argument"};
        *logits = s->impl->host_logits;
    });
}

gh_status gh_session_prefill(gh_session* sess, const int32_t* ids, int32_t len,
                             float* last_logits_host) {
    return guard([&] {
        if (!sess || !ids) throw ApiError{GH_ERR_INVALID_ARGUMENT, "null argument"};
        Session& s = *sess->impl;
        const PersistGate gate(s);  // held until this call has synchronised its launches
        const ResidentScope scope(s);
        if (len < 0) throw ApiError{GH_ERR_INVALID_ARGUMENT, "negative length"};
        if (len == 0) return;
        if (s.pos + len > s.m->shape.max_len)
            throw ApiError{GH_ERR_RUNTIME, "InferenceSession: context exceeds max_len"};
        check_ids(s, ids, static_cast<size_t>(s.B) * len);
        const size_t V = s.m->shape.vocab;
        // Stage the ids into the history, then step through them.
        std::memcpy(s.host_ids, ids, static_cast<size_t>(s.B) * len * sizeof(int));
        stage_ids(s, s.host_ids, len, s.hist, s.hist_stride, s.n_hist);
        run_resident(s, [&] {
            run_prompt(s, len, nullptr, nullptr);
            deliver_logits(s);
            HIP_CHECK(hipStreamSynchronize(s.stream));
        });
        check_persist_abort(s);
        if (last_logits_host) std::memcpy(last_logits_host, s.host_logits, s.B * V * sizeof(float));
    });
}

gh_status gh_session_score(gh_session* sess, const int32_t* ids, const int32_t* targets, int32_t len,
                           float* nll_host) {
    return guard([&] {
        if (!sess || !ids || !targets || !nll_host) throw ApiError{GH_ERR_INVALID_ARGUMENT, "null argument"};
        Session& s = *sess->impl;
        const PersistGate gate(s);  // held until this call has synchronised its launches
        const ResidentScope scope(s);
        if (len < 0) throw ApiError{GH_ERR_INVALID_ARGUMENT, "negative length"};
        if (len == 0) return;
        if (s.pos + len > s.m->shape.max_len)
            throw ApiError{GH_ERR_RUNTIME, "InferenceSession: context exceeds max_len"};
        const size_t n = static_cast<size_t>(s.B) * len;
        check_ids(s, ids, n);
        check_ids(s, targets, n);
        const int base = s.n_hist;
        int* host_targets = s.host_ids + static_cast<size_t>(s.B) * s.hist_stride;
        std::memcpy(s.host_ids, ids, n * sizeof(int));
        std::memcpy(host_targets, targets, n * sizeof(int));
        stage_ids(s, s.host_ids, len, s.hist, s.hist_stride, base);
        if (s.score_cap < n) {
            if (s.score_targets) HIP_CHECK(hipFree(s.score_targets));
            if (s.score_nll) HIP_CHECK(hipFree(s.score_nll));
            s.score_targets = nullptr;
            s.score_nll = nullptr;
            s.score_cap = 0;
            dev_alloc(s.score_targets, n);
            dev_alloc(s.score_nll, n);
            s.score_cap = n;
        }
        stage_ids(s, host_targets, len, s.score_targets, len, 0);
        const ScoreSink sink{s.score_targets, s.score_nll};
        const RowsPlan plan = plan_rows(s, len, /*score=*/true);
        run_resident(s, [&] {
            if (plan.slice > 0) {
                prompt_pass(s, len, plan, &sink);
            } else {
                // token by token: every step leaves the logits of its position
                const int V = s.m->shape.vocab;
                for (int t = 0; t < len; t++) {
                    if (s.engine == GH_ENGINE_PERSISTENT) {
                        persist_run(s, 1, 1, 0, false, nullptr, nullptr, 0, 0, nullptr);  // token from the history
                    } else {
                        hipLaunchKernelGGL(load_tok_kernel, dim3((s.B + 63) / 64), dim3(64), 0, s.stream, s.hist,
                                           s.hist_stride, base + t, s.tok, s.B);
                        HIP_CHECK(hipGetLastError());
                        run_step(s);
                    }
                    hipLaunchKernelGGL(nll_rows_kernel, dim3(s.B), dim3(256), 0, s.stream, s.logits, V, t, len, sink.targets,
                                       sink.nll);
                    HIP_CHECK(hipGetLastError());
                }
                if (s.engine != GH_ENGINE_PERSISTENT) s.n_hist += len;
            }
            deliver(s, s.score_nll, 0, 1, n, s.host_ids);  // (the ids have long been read)
            HIP_CHECK(hipStreamSynchronize(s.stream));
        });
        check_persist_abort(s);
        std::memcpy(nll_host, s.host_ids, n * sizeof(float));
    });
}

int32_t gh_session_position(const gh_session* s) { return s ? s->impl->pos : -1; }
int32_t gh_session_capacity(const gh_session* s) { return s ? s->impl->m->shape.max_len : -1; }
int32_t gh_session_vocab(const gh_session* s) { return s ? s->impl->m->shape.vocab : -1; }
int32_t gh_session_batch(const gh_session* s) { return s ? s->impl->B : -1; }

gh_status gh_session_read_kv(gh_session* sess, int32_t seq, int32_t layer, int32_t kv, int32_t pos,
                             float* out_host) {
    return guard([&] {
        if (!sess || !out_host) throw ApiError{GH_ERR_INVALID_ARGUMENT, "null argument"};
        Session& s = *sess->impl;
        const Shape& sh = s.m->shape;
        if (seq < 0 || seq >= s.B || layer < 0 || layer >= sh.layers || kv < 0 || kv > 1 || pos < 0
            || pos >= s.pos)
            throw ApiError{GH_ERR_OUT_OF_RANGE, "cache row out of range"};
        HIP_CHECK(hipStreamSynchronize(s.stream));
        std::vector<int> table(static_cast<size_t>(s.n_pages));
        HIP_CHECK(hipMemcpy(table.data(), s.page_table, table.size() * sizeof(int),
                            hipMemcpyDeviceToHost));
        const int hs = sh.head_size();
        const int page = table[static_cast<size_t>(seq) * s.pages_per_seq + (pos >> s.page_shift)];
        const int slot = pos & ((1 << s.page_shift) - 1);
        for (int h = 0; h < sh.heads; h++) {
            const size_t run = ((static_cast<size_t>(layer) * s.n_pages + page) * 2 + kv) * sh.heads + h;
            const size_t off = ((run << s.page_shift) + slot) * hs;
            HIP_CHECK(hipMemcpy(out_host + static_cast<size_t>(h) * hs, s.kv_pool + off,
                                hs * sizeof(float), hipMemcpyDeviceToHost));
        }
    });
}

gh_status gh_session_pick(gh_session* sess, const gh_sampling* opt, const float* uniforms,
                          uint64_t seed, int32_t* out_ids) {
    return guard([&] {
        if (!sess || !opt) throw ApiError{GH_ERR_INVALID_ARGUMENT, "null argument"};
        Session& s = *sess->impl;
        check_sampling(*opt);
        if (s.pos == 0) throw ApiError{GH_ERR_RUNTIME, "no logits yet: step or prefill first"};
        if (s.n_hist >= s.hist_stride)
            throw ApiError{GH_ERR_RUNTIME, "token history is full"};
        const float* du = nullptr;
        if (uniforms) {
            if (s.uniforms_cap < static_cast<size_t>(s.B)) {
                if (s.uniforms) HIP_CHECK(hipFree(s.uniforms));
                s.uniforms = nullptr;
                dev_alloc(s.uniforms, s.B);
                s.uniforms_cap = s.B;
            }
            HIP_CHECK(hipMemcpyAsync(s.uniforms, uniforms, s.B * sizeof(float),
                                     hipMemcpyHostToDevice, s.stream));
            du = s.uniforms;
        }
        // The draw index is folded into the pointer: one uniform per sequence here.
        const int saved = s.picks;
        if (du) s.picks = 0;
        launch_pick(s, *opt, du, 1, seed, false);  // the stand-alone pick kernel serves every engine
        if (du) s.picks = saved + 1;
        deliver(s, s.tok, 0, 1, s.B, s.host_ids);
        HIP_CHECK(hipStreamSynchronize(s.stream));
        if (out_ids) std::memcpy(out_ids, s.host_ids, s.B * sizeof(int));
    });
}

gh_status gh_session_decode(gh_session* sess, int32_t max_tokens, const gh_sampling* opt,
                            const float* uniforms, uint64_t seed, int32_t* out_ids,
                            int32_t* out_count) {
    return guard([&] {
        if (!sess || !opt || !out_count) throw ApiError{GH_ERR_INVALID_ARGUMENT, "null argument"};
        Session& s = *sess->impl;
        const PersistGate gate(s);  // held until this call has synchronised its launches
        const ResidentScope scope(s);
        check_sampling(*opt);
        *out_count = 0;
        s.timing = gh_timing{};
        s.timing.launches_per_step = s.launches_per_step;
        if (max_tokens <= 0) return;
        if (s.pos == 0) throw ApiError{GH_ERR_RUNTIME, "no logits yet: step or prefill first"};
        const size_t B = s.B;
        const float* du = opt->greedy ? nullptr : stage_uniforms(s, uniforms, B * max_tokens);
        const int first = s.n_hist;
        const int saved_picks = s.picks;
        if (du) s.picks = 0;  // uniforms are indexed from this call's first pick
        int made = 0, stepped = 0;
        bool again = false;
        keep_logits(s, /*restore=*/false);
        run_resident(s, [&] {
            if (again) keep_logits(s, /*restore=*/true);
            again = true;
            HIP_CHECK(hipEventRecord(s.ev[1], s.stream));
            std::tie(made, stepped) = run_decode(s, max_tokens, *opt, du, max_tokens, seed, nullptr, nullptr);
            HIP_CHECK(hipEventRecord(s.ev[2], s.stream));
            deliver(s, s.hist + first, s.hist_stride, s.B, made, s.host_ids);
            HIP_CHECK(hipStreamSynchronize(s.stream));
        });
        if (du) s.picks = saved_picks + made;
        check_persist_abort(s);
        if (out_ids)
            for (size_t b = 0; b < B; b++)
                std::memcpy(out_ids + b * max_tokens, s.host_ids + b * made, made * sizeof(int));
        *out_count = made;
        HIP_CHECK(hipEventElapsedTime(&s.timing.decode_ms, s.ev[1], s.ev[2]));
        s.timing.decode_steps = stepped;
        s.timing.launches_per_step = s.launches_per_step;
    });
}

gh_status gh_session_decode_stream(gh_session* sess, int32_t max_tokens, const gh_sampling* opt,
                                   const float* uniforms, uint64_t seed, int32_t stop_token,
                                   gh_token_callback on_tokens, void* user, int32_t* out_ids,
                                   int32_t* out_count) {
    return guard([&] {
        if (!sess || !opt || !out_count || !on_tokens) throw ApiError{GH_ERR_INVALID_ARGUMENT, "null argument"};
        Session& s = *sess->impl;
        const PersistGate gate(s);  // held until this call has synchronised its launches
        const ResidentScope scope(s);
        check_sampling(*opt);
        *out_count = 0;
        s.timing = gh_timing{};
        s.timing.launches_per_step = s.launches_per_step;
        if (max_tokens <= 0) return;
        if (s.pos == 0) throw ApiError{GH_ERR_RUNTIME, "no logits yet: step or prefill first"};
        const int B = s.B, C = s.m->shape.max_len;
        const float* du = opt->greedy ? nullptr : stage_uniforms(s, uniforms, static_cast<size_t>(B) * max_tokens);
        const int saved_picks = s.picks;
        if (du) s.picks = 0;  // uniforms are indexed from this call's first pick
        int made = 0, stepped = 0;
        HIP_CHECK(hipEventRecord(s.ev[1], s.stream));
        if (s.engine == GH_ENGINE_PERSISTENT) {
            // One launch runs the whole loop; the kernel reports each pick in pinned
            // memory as it is made and this thread hands it on while the kernel goes on.
            int planned_picks = 0, planned_steps = 0, pos = s.pos, nh = s.n_hist;
            for (int i = 0; i < max_tokens; i++) {
                if (nh >= s.hist_stride) break;
                planned_picks++;
                nh++;
                if (pos >= C) break;
                planned_steps++;
                pos++;
            }
            __atomic_store_n(s.stop_word, 0u, __ATOMIC_RELEASE);
            const unsigned base = s.feed_base;
            persist_run(s, 0, planned_steps, planned_picks, true, opt, du, max_tokens, seed, nullptr, true,
                        stop_token);
            HIP_CHECK(hipEventRecord(s.ev[2], s.stream));
            bool kernel_done = false;
            unsigned idle = 0;
            // Whatever ends this loop (the callback, a HIP error), the kernel must have
            // stopped and the host's view must match the device's before control leaves.
            auto settle = [&] {
                stepped = std::min(made, planned_steps);
                s.pos -= planned_steps - stepped;
                s.arrive_total -= static_cast<unsigned>(planned_steps - stepped);
                s.n_hist -= planned_picks - made;
                s.picks -= planned_picks - made;
            };
            try {
                while (made < planned_picks) {
                    const unsigned long long w = __atomic_load_n(s.feed + made, __ATOMIC_ACQUIRE);
                    if (static_cast<unsigned>(w >> 32) == base + static_cast<unsigned>(made) + 1u) {
                        const int32_t tok = static_cast<int32_t>(static_cast<unsigned>(w));
                        if (tok < 0) break;  // the kernel saw the stop word before this pick
                        if (out_ids) out_ids[made] = tok;
                        made++;  // delivered (or thrown out of) below: the round counts either way
                        const int32_t asked = on_tokens(user, &tok, made - 1);
                        idle = 0;
                        if (asked != 0) __atomic_store_n(s.stop_word, 1u, __ATOMIC_RELEASE);
                        if (tok == stop_token) break;  // the kernel ends after this token's step
                        continue;
                    }
                    if (kernel_done) break;  // the launch is over and reported no further pick
                    if ((++idle & 255u) == 0u) {
                        const hipError_t q = hipStreamQuery(s.stream);
                        if (q == hipSuccess) kernel_done = true;  // read the feed once more, then leave
                        else if (q != hipErrorNotReady) HIP_CHECK(q);
                    }
                }
            } catch (...) {
                // stop the kernel at its next pick, wait for it, and take every round it
                // still completed into account before handing the error on
                __atomic_store_n(s.stop_word, 1u, __ATOMIC_RELEASE);
                (void)hipStreamSynchronize(s.stream);
                while (made < planned_picks) {
                    const unsigned long long w = __atomic_load_n(s.feed + made, __ATOMIC_ACQUIRE);
                    if (static_cast<unsigned>(w >> 32) != base + static_cast<unsigned>(made) + 1u
                        || static_cast<int32_t>(static_cast<unsigned>(w)) < 0)
                        break;
                    if (out_ids) out_ids[made] = static_cast<int32_t>(static_cast<unsigned>(w));
                    made++;
                }
                settle();
                if (du) s.picks = saved_picks + made;
                *out_count = made;
                throw;
            }
            deliver(s, nullptr, 0, 1, 0, nullptr);
            HIP_CHECK(hipStreamSynchronize(s.stream));
            check_persist_abort(s);
            // persist_run advanced the host's view by the planned run: take back what was not run
            settle();
        } else {
            std::vector<char> seen(static_cast<size_t>(B), 0);
            int n_seen = 0;
            for (int i = 0; i < max_tokens; i++) {
                if (s.n_hist >= s.hist_stride) break;
                launch_pick(s, *opt, du, max_tokens, seed, true, /*embed=*/s.pos < C);
                deliver(s, s.tok, 0, 1, B, s.host_ids);
                HIP_CHECK(hipStreamSynchronize(s.stream));
                resident_end(s);  // the callback may use any session
                if (repeat_step(s, /*picked=*/true)) {
                    i--;  // its pick was made from nothing
                    continue;
                }
                if (out_ids)
                    for (int b = 0; b < B; b++) out_ids[static_cast<size_t>(b) * max_tokens + i] = s.host_ids[b];
                const int32_t asked = on_tokens(user, s.host_ids, i);
                made++;
                for (int b = 0; b < B; b++)
                    if (s.host_ids[b] == stop_token && !seen[b]) {
                        seen[b] = 1;
                        n_seen++;
                    }
                if (s.pos >= C) break;
                run_step(s, STEP_ROWS);
                stepped++;
                if (asked != 0 || n_seen == B) break;
            }
            HIP_CHECK(hipEventRecord(s.ev[2], s.stream));
            if (s.resident) deliver(s, nullptr, 0, 1, 0, nullptr);
            HIP_CHECK(hipStreamSynchronize(s.stream));
            if (repeat_step(s, /*picked=*/false)) HIP_CHECK(hipStreamSynchronize(s.stream));
        }
        if (du) s.picks = saved_picks + made;
        *out_count = made;
        HIP_CHECK(hipEventElapsedTime(&s.timing.decode_ms, s.ev[1], s.ev[2]));
        s.timing.decode_steps = stepped;
        s.timing.launches_per_step = s.launches_per_step;
    });
}

gh_status gh_session_generate(gh_session* sess, const int32_t* prompts, int32_t prompt_len,
                              int32_t max_tokens, const gh_sampling* opt, const float* uniforms,
                              uint64_t seed, int32_t* out_tokens, int32_t* out_len,
                              float* step_logits_host, int32_t* n_steps) {
    return guard([&] {
        if (!sess || !opt || !out_tokens || !out_len)
            throw ApiError{GH_ERR_INVALID_ARGUMENT, "null argument"};
        Session& s = *sess->impl;
        const PersistGate gate(s);  // held until this call has synchronised its launches
        const ResidentScope scope(s);
        const Shape& sh = s.m->shape;
        check_sampling(*opt);
        *out_len = 0;
        if (n_steps) *n_steps = 0;
        s.timing = gh_timing{};
        s.timing.launches_per_step = s.launches_per_step;
        if (prompt_len <= 0) return;  // text_gen.cpp:40: an empty prompt generates nothing
        if (!prompts) throw ApiError{GH_ERR_INVALID_ARGUMENT, "null prompts"};
        if (max_tokens < 0) max_tokens = 0;
        check_ids(s, prompts, static_cast<size_t>(s.B) * prompt_len);
        if (prompt_len > sh.max_len)
            throw ApiError{GH_ERR_RUNTIME, "InferenceSession: context exceeds max_len"};
        const size_t B = s.B, V = sh.vocab;

        reset_session(s);
        std::memcpy(s.host_ids, prompts, B * prompt_len * sizeof(int));
        stage_ids(s, s.host_ids, prompt_len, s.hist, s.hist_stride, 0);
        const float* du =
            opt->greedy ? nullptr : stage_uniforms(s, uniforms, B * static_cast<size_t>(max_tokens));
        float* log = nullptr;
        if (step_logits_host) {
            const size_t need = (static_cast<size_t>(prompt_len) + max_tokens) * B * V;
            if (s.logit_log_cap < need) {
                if (s.logit_log) HIP_CHECK(hipFree(s.logit_log));
                s.logit_log = nullptr;
                dev_alloc(s.logit_log, need);
                s.logit_log_cap = need;
            }
            log = s.logit_log;
        }
        size_t steps = 0;
        int made = 0, stepped = 0, total = 0;
        run_resident(s, [&] {
            steps = 0;
            HIP_CHECK(hipEventRecord(s.ev[0], s.stream));
            run_prompt(s, prompt_len, log, &steps);
            HIP_CHECK(hipEventRecord(s.ev[1], s.stream));
            s.ahead = Session::AHEAD_PROMPT;
            std::tie(made, stepped) = run_decode(s, max_tokens, *opt, du, max_tokens, seed, log, &steps);
            HIP_CHECK(hipEventRecord(s.ev[2], s.stream));

            total = s.n_hist;
            deliver(s, s.hist, s.hist_stride, s.B, total, s.host_ids);
            HIP_CHECK(hipStreamSynchronize(s.stream));
        });
        check_persist_abort(s);
        const size_t out_stride = static_cast<size_t>(prompt_len) + max_tokens;
        for (size_t b = 0; b < B; b++)
            std::memcpy(out_tokens + b * out_stride, s.host_ids + b * total, total * sizeof(int));
        *out_len = total;
        if (step_logits_host)
            HIP_CHECK(hipMemcpy(step_logits_host, s.logit_log, steps * B * V * sizeof(float),
                                hipMemcpyDeviceToHost));
        if (n_steps) *n_steps = static_cast<int32_t>(steps);
        HIP_CHECK(hipEventElapsedTime(&s.timing.prompt_ms, s.ev[0], s.ev[1]));
        HIP_CHECK(hipEventElapsedTime(&s.timing.decode_ms, s.ev[1], s.ev[2]));
        s.timing.prompt_steps = prompt_len;
        s.timing.decode_steps = stepped;
        s.timing.launches_per_step = s.launches_per_step;
    });
}

gh_status gh_pick_noalloc(const float* logits, int32_t batch, int32_t vocab, const int32_t* history,
                          int32_t history_stride, int32_t n_history, const gh_sampling* opt,
                          const float* uniforms, uint64_t seed, int32_t pick_index, int32_t* out_ids,
                          void* hip_stream) {
    return guard([&] {
        if (!logits || !opt || !out_ids) throw ApiError{GH_ERR_INVALID_ARGUMENT, "null argument"};
        if (batch < 1 || vocab < 1 || n_history < 0 || pick_index < 0 || n_history > history_stride
            || (n_history > 0 && !history))
            throw ApiError{GH_ERR_INVALID_ARGUMENT, "gh_pick_noalloc: bad sizes"};
        check_sampling(*opt);
        const size_t work_stride = (static_cast<size_t>(vocab) + kPickThreads + 3) / 4 * 4;
        if (static_cast<size_t>(batch) * work_stride > kNoAllocScratchFloats)
            throw ApiError{GH_ERR_INVALID_ARGUMENT,
                           "gh_pick_noalloc: batch x (vocab + 1024) floats exceed the 4 MiB scratch array ("
                               + std::to_string(kNoAllocScratchFloats) + " floats)"};
        PickParams p{};
        p.logits = logits;
        p.work = scratch_on_current_device();
        p.work_stride = static_cast<int>(work_stride);
        p.V = vocab;
        p.hist = const_cast<int*>(history);  // read only on this path
        p.hist_stride = history_stride;
        p.n_hist = n_history;
        p.pick_idx = uniforms ? 0 : pick_index;
        p.tok = nullptr;
        p.temperature = opt->temperature;
        p.top_k = opt->top_k;
        p.top_p = opt->top_p;
        p.penalty = opt->repetition_penalty;
        p.greedy = opt->greedy;
        p.uniforms = uniforms;
        p.u_stride = 1;
        p.seed_lo = static_cast<unsigned>(seed & 0xFFFFFFFFu);
        p.seed_hi = static_cast<unsigned>(seed >> 32);
        p.sort_cap = kPickWorkFloats;
        hipLaunchKernelGGL(pick_noalloc_kernel, dim3(batch), dim3(kPickThreads), kPickWorkFloats * sizeof(float),
                           static_cast<hipStream_t>(hip_stream), p, out_ids);
        HIP_CHECK(hipGetLastError());
    });
}

gh_status gh_session_last_timing(const gh_session* s, gh_timing* out) {
    return guard([&] {
        if (!s || !out) throw ApiError{GH_ERR_INVALID_ARGUMENT, "null argument"};
        *out = s->impl->timing;
        out->row_picks = 0;
        if (s->impl->ctl) {
            unsigned n = 0;
            HIP_CHECK(hipMemcpy(&n, &s->impl->ctl->row_picks, sizeof(n), hipMemcpyDeviceToHost));
            out->row_picks = static_cast<int32_t>(n);
        }
    });
}

gh_status gh_device_info(char* name, size_t name_len, int32_t* compute_units, int32_t* is_gfx950) {
    return guard([&] {
        require_gpu();
        int dev = 0;
        HIP_CHECK(hipGetDevice(&dev));
        hipDeviceProp_t prop;
        HIP_CHECK(hipGetDeviceProperties(&prop, dev));
        if (name && name_len) {
            std::snprintf(name, name_len, "%s (%s)", prop.name, prop.gcnArchName);
        }
        if (compute_units) *compute_units = prop.multiProcessorCount;
        if (is_gfx950) *is_gfx950 = std::strstr(prop.gcnArchName, "gfx950") != nullptr;
        (void)scratch_on_current_device();  // set-up for gh_pick_noalloc on this device
    });
}

gh_status gh_device_read_bandwidth(size_t bytes, int32_t repeats, double* gb_per_s) {
    return guard([&] {
        require_gpu();
        if (!gb_per_s || bytes < (1u << 20) || repeats < 1)
            throw ApiError{GH_ERR_INVALID_ARGUMENT, "read bandwidth probe: need >= 1 MiB, >= 1 repeat"};
        const size_t n4 = bytes / sizeof(float4);
        struct Scratch {  // released on every path out of this function
            float4* buf = nullptr;
            float* sink = nullptr;
            hipEvent_t e0 = nullptr, e1 = nullptr;
            ~Scratch() {
                if (e0) (void)hipEventDestroy(e0);
                if (e1) (void)hipEventDestroy(e1);
                if (buf) (void)hipFree(buf);
                if (sink) (void)hipFree(sink);
            }
        } t;
        HIP_CHECK(hipMalloc(&t.buf, n4 * sizeof(float4)));
        HIP_CHECK(hipMalloc(&t.sink, sizeof(float)));
        HIP_CHECK(hipMemset(t.buf, 0x3c, n4 * sizeof(float4)));  // finite floats, not zeros
        HIP_CHECK(hipEventCreate(&t.e0));
        HIP_CHECK(hipEventCreate(&t.e1));
        double best = 0.0;
        for (int r = 0; r < repeats + 1; r++) {  // the first pass warms up
            HIP_CHECK(hipEventRecord(t.e0, nullptr));
            hipLaunchKernelGGL(stream_read_kernel, dim3(8192), dim3(256), 0, nullptr, t.buf, n4, t.sink);
            HIP_CHECK(hipGetLastError());
            HIP_CHECK(hipEventRecord(t.e1, nullptr));
            HIP_CHECK(hipEventSynchronize(t.e1));
            float ms = 0.0f;
            HIP_CHECK(hipEventElapsedTime(&ms, t.e0, t.e1));
            if (r > 0) best = std::max(best, static_cast<double>(n4) * sizeof(float4) / (ms * 1e-3) / 1e9);
        }
        *gb_per_s = best;
    });
}

gh_status gh_device_handoff_latency(int32_t load_policy, int32_t device_scope_store, int32_t peer, int32_t busy,
                                    double* us_per_round_trip, int32_t* xcd_a, int32_t* xcd_b) {
    return guard([&] {
        require_gpu();
        HandoffKernel kernel = handoff_kernel_for(load_policy, device_scope_store != 0);
        if (!kernel || !us_per_round_trip || peer < 1 || peer > 15)
            throw ApiError{GH_ERR_INVALID_ARGUMENT, "hand-off probe: load policy 0..2, peer workgroup 1..15"};
        struct Scratch {  // released on every path out of this function
            unsigned *cells = nullptr, *xcds = nullptr, *stop = nullptr;
            unsigned long long* ticks = nullptr;
            float4* big = nullptr;
            float* sink = nullptr;
            hipStream_t s1 = nullptr, s2 = nullptr;
            ~Scratch() {
                if (stop) *stop = 1u;
                (void)hipDeviceSynchronize();
                if (s1) (void)hipStreamDestroy(s1);
                if (s2) (void)hipStreamDestroy(s2);
                for (void* p : {static_cast<void*>(cells), static_cast<void*>(xcds), static_cast<void*>(ticks),
                                static_cast<void*>(big), static_cast<void*>(sink)})
                    if (p) (void)hipFree(p);
                if (stop) (void)hipHostFree(stop);
            }
        } t;
        const int rounds = 1000;
        const size_t big_bytes = busy ? (size_t(2) << 30) : sizeof(float4);
        dev_alloc(t.cells, 256);
        dev_alloc(t.xcds, 16);
        dev_alloc(t.ticks, 2);
        HIP_CHECK(hipMalloc(&t.big, big_bytes));
        HIP_CHECK(hipMemset(t.big, 0, big_bytes));
        dev_alloc(t.sink, 1);
        HIP_CHECK(hipHostMalloc(&t.stop, sizeof(unsigned), hipHostMallocCoherent));
        *t.stop = 0u;
        HIP_CHECK(hipStreamCreateWithFlags(&t.s1, hipStreamNonBlocking));
        HIP_CHECK(hipStreamCreateWithFlags(&t.s2, hipStreamNonBlocking));
        HIP_CHECK(hipDeviceSynchronize());
        if (busy) {
            hipLaunchKernelGGL(handoff_probe_hog, dim3(240), dim3(256), 0, t.s2, t.big, big_bytes / sizeof(float4),
                               t.stop, t.sink);
            HIP_CHECK(hipGetLastError());
        }
        hipLaunchKernelGGL(kernel, dim3(16), dim3(64), 0, t.s1, t.cells, peer, rounds, t.ticks, t.xcds);
        HIP_CHECK(hipGetLastError());
        HIP_CHECK(hipStreamSynchronize(t.s1));
        *t.stop = 1u;
        HIP_CHECK(hipDeviceSynchronize());
        unsigned long long ticks[2];
        unsigned xcds[16];
        HIP_CHECK(hipMemcpy(ticks, t.ticks, sizeof(ticks), hipMemcpyDeviceToHost));
        HIP_CHECK(hipMemcpy(xcds, t.xcds, sizeof(xcds), hipMemcpyDeviceToHost));
        *us_per_round_trip = static_cast<double>(ticks[0]) / 100.0 / rounds;
        if (xcd_a) *xcd_a = static_cast<int32_t>(xcds[0]);
        if (xcd_b) *xcd_b = static_cast<int32_t>(xcds[peer]);
    });
}

gh_status gh_device_mfma_issue(int32_t mode, int32_t valu_per_slot, double* clk_per_product, double* clk_per_valu_slot,
                               double* shader_mhz) {
    return guard([&] {
        require_gpu();
        using Kernel = void (*)(long long*, int, int, float, float);
        Kernel kernel = valu_per_slot == 8    ? mfma_issue_probe_kernel<8>
                        : valu_per_slot == 16 ? mfma_issue_probe_kernel<16>
                        : valu_per_slot == 24 ? mfma_issue_probe_kernel<24>
                                              : nullptr;
        if (!kernel || mode < 1 || mode > 6 || (mode & 1 && mode & 4) || !clk_per_product || !clk_per_valu_slot ||
            !shader_mhz)
            throw ApiError{GH_ERR_INVALID_ARGUMENT, "matrix-core issue probe: mode 1, 2, 3, 4 or 6; 8, 16 or 24 "
                                                    "multiply-adds per slot"};
        const int blocks = 256, iters = 4000;
        struct Scratch {
            long long* out = nullptr;
            ~Scratch() {
                if (out) (void)hipFree(out);
            }
        } t;
        dev_alloc(t.out, static_cast<size_t>(blocks) * 8 * 3);
        for (int rep = 0; rep < 2; rep++) {  // the first run brings the clock up
            hipLaunchKernelGGL(kernel, dim3(blocks), dim3(512), 0, nullptr, t.out, iters, mode, 1.0f, 0.999f);
            HIP_CHECK(hipGetLastError());
            HIP_CHECK(hipDeviceSynchronize());
        }
        std::vector<long long> h(static_cast<size_t>(blocks) * 8 * 3);
        HIP_CHECK(hipMemcpy(h.data(), t.out, h.size() * sizeof(long long), hipMemcpyDeviceToHost));
        double mfma = 0.0, valu = 0.0, cyc = 0.0, wall = 0.0;
        for (int b = 0; b < blocks; b++)
            for (int w = 0; w < 8; w++) {
                const long long* o = &h[(static_cast<size_t>(b) * 8 + w) * 3];
                (w < 4 ? mfma : valu) += static_cast<double>(o[0]);
                const bool busy = w < 4 ? (mode & 5) != 0 : (mode & 2) != 0;
                if (busy) {
                    cyc += static_cast<double>(o[0]);
                    wall += static_cast<double>(o[1]);
                }
            }
        const double slots = static_cast<double>(blocks) * 4 * iters * 8;
        *clk_per_product = (mode & 5) ? mfma / slots : 0.0;
        *clk_per_valu_slot = (mode & 2) ? valu / slots : 0.0;
        *shader_mhz = wall > 0.0 ? cyc / wall * 100.0 : 0.0;  // the constant clock counts at 100 MHz
    });
}

gh_status gh_device_reread_bandwidth(size_t bytes, int32_t passes, double* gb_per_s) {
    return guard([&] {
        require_gpu();
        if (!gb_per_s || bytes < (1u << 20) || passes < 1)
            throw ApiError{GH_ERR_INVALID_ARGUMENT, "re-read bandwidth probe: need >= 1 MiB, >= 1 pass"};
        const size_t n4 = bytes / sizeof(float4);
        struct Scratch {
            float4* buf = nullptr;
            float* sink = nullptr;
            hipEvent_t e0 = nullptr, e1 = nullptr;
            ~Scratch() {
                if (e0) (void)hipEventDestroy(e0);
                if (e1) (void)hipEventDestroy(e1);
                if (buf) (void)hipFree(buf);
                if (sink) (void)hipFree(sink);
            }
        } t;
        HIP_CHECK(hipMalloc(&t.buf, n4 * sizeof(float4)));
        HIP_CHECK(hipMalloc(&t.sink, sizeof(float)));
        HIP_CHECK(hipMemset(t.buf, 0x3c, n4 * sizeof(float4)));  // finite floats, not zeros
        HIP_CHECK(hipEventCreate(&t.e0));
        HIP_CHECK(hipEventCreate(&t.e1));
        // Every pass is a launch of its own that streams the whole buffer (passes inside one
        // launch would only re-read what the resident workgroups hold, which the L2s serve).
        // 2048 x 256 threads with eight loads each cover 64 MiB per round.
        const int grid = static_cast<int>(std::min<size_t>(8192, std::max<size_t>(256, n4 / (256 * 8))));
        for (int r = -2; r < passes; r++) {  // two passes warm up, then one span over the rest
            if (r == 0) HIP_CHECK(hipEventRecord(t.e0, nullptr));
            hipLaunchKernelGGL(stream_read_kernel, dim3(grid), dim3(256), 0, nullptr, t.buf, n4, t.sink);
        }
        HIP_CHECK(hipGetLastError());
        HIP_CHECK(hipEventRecord(t.e1, nullptr));
        HIP_CHECK(hipEventSynchronize(t.e1));
        float ms = 0.0f;
        HIP_CHECK(hipEventElapsedTime(&ms, t.e0, t.e1));
        *gb_per_s = static_cast<double>(passes) * static_cast<double>(n4) * sizeof(float4) / (ms * 1e-3) / 1e9;
    });
}

}  // extern "C"
