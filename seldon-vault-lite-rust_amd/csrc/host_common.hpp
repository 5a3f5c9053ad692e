// Host-side helpers shared by the text runtime (runtime.cpp) and the vision
// runtime (vision.cpp): the thread-local error message, status macros,
// growable device buffers, and weight-inventory validation / decoding in the
// manner of src/model/weights.rs:125-189 and src/binary/safetensors.rs:69-110.
#pragma once

#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <map>
#include <string>
#include <utility>
#include <vector>

#include "../../include/svl_hip.h"
#include "svl_internal.hpp"

struct svl_ctx {
    int device;
};

namespace svl {

inline thread_local std::string g_err;

inline svl_status fail(svl_status st, const char *fmt, ...) {
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof buf, fmt, ap);
    va_end(ap);
    g_err = buf;
    return st;
}

#define HIP_TRY(expr)                                                                       \
    do {                                                                                    \
        hipError_t e_ = (expr);                                                             \
        if (e_ != hipSuccess) return fail(SVL_DEVICE, "%s: %s", #expr, hipGetErrorString(e_)); \
    } while (0)

#define ST_TRY(expr)                    \
    do {                                \
        svl_status s_ = (expr);         \
        if (s_ != SVL_OK) return s_;    \
    } while (0)

// src/tensor/owned.rs MAX_TENSOR_ELEMENTS, text.rs:34 MAX_ACTIVATION_ELEMENTS.
constexpr int64_t MAX_ACTIVATION_ELEMENTS = int64_t(1) << 28;
constexpr int64_t MAX_TENSOR_ELEMENTS = int64_t(1) << 30;

template <class T>
struct DevBuf {
    T *p = nullptr;
    size_t n = 0;
    hipError_t ensure(size_t count) {
        if (count <= n) return hipSuccess;
        if (p) (void)hipFree(p);
        p = nullptr;
        n = 0;
        hipError_t e = hipMalloc((void **)&p, std::max<size_t>(count, 1) * sizeof(T));
        if (e == hipSuccess) n = count;
        return e;
    }
    void release() {
        if (p) (void)hipFree(p);
        p = nullptr;
        n = 0;
    }
};

using ShapeList = std::vector<std::pair<std::string, std::vector<int64_t>>>;
using TensorIndex = std::map<std::string, const svl_tensor_view *>;

// Inventory check of a weight set (weights.rs:130-165, vision.rs:556-594):
// a tensor under one of `prefixes` that the shape list does not name is
// unexpected (CORRUPT), a named tensor that is absent or mis-shaped is
// CORRUPT, and the per-tensor and total element caps give LIMIT.
inline svl_status check_inventory(const svl_tensor_view *tensors, size_t n_tensors,
                                  const ShapeList &shapes,
                                  std::initializer_list<const char *> prefixes, const char *kind,
                                  int64_t max_total, TensorIndex &by_name) {
    by_name.clear();
    for (size_t i = 0; i < n_tensors; ++i) {
        if (!tensors[i].name) return fail(SVL_USAGE, "tensor %zu has no name", i);
        by_name[tensors[i].name] = &tensors[i];
    }
    std::map<std::string, size_t> expected;
    for (size_t i = 0; i < shapes.size(); ++i) expected[shapes[i].first] = i;
    for (auto &kv : by_name) {
        bool ours = false;
        for (const char *p : prefixes) ours = ours || kv.first.rfind(p, 0) == 0;
        if (ours && !expected.count(kv.first))
            return fail(SVL_CORRUPT, "unexpected %s tensor %s in the weight file", kind,
                        kv.first.c_str());
    }
    int64_t parameters = 0;
    for (auto &sh : shapes) {
        auto it = by_name.find(sh.first);
        if (it == by_name.end())
            return fail(SVL_CORRUPT, "%s weight %s is missing from the Safetensors file", kind,
                        sh.first.c_str());
        const svl_tensor_view *t = it->second;
        bool same = t->ndim == (int32_t)sh.second.size();
        for (size_t d = 0; same && d < sh.second.size(); ++d) same = t->shape[d] == sh.second[d];
        if (!same)
            return fail(SVL_CORRUPT, "%s weight %s has an unexpected shape", kind, sh.first.c_str());
        int64_t numel = 1;
        for (int64_t d : sh.second) numel *= d;
        if (numel > MAX_TENSOR_ELEMENTS)
            return fail(SVL_LIMIT, "tensor %s has %lld elements, above the cap", sh.first.c_str(),
                        (long long)numel);
        parameters += numel;
        if (parameters > max_total)
            return fail(SVL_LIMIT, "%s weights exceed the %lld-element cap", kind,
                        (long long)max_total);
        if (!t->data) return fail(SVL_USAGE, "tensor %s has no data", sh.first.c_str());
    }
    return SVL_OK;
}

// TensorEntry::to_f32 (safetensors.rs:69-110): F32 little-endian or BF16
// widened exactly (bf16.rs:13-15, bits << 16), each after the payload length
// check of the reference (safetensors.rs:79-88, bf16.rs:40-51). numel is at
// most MAX_TENSOR_ELEMENTS, so the byte counts cannot overflow. Non-finite
// values are rejected like Tensor::validate_finite (owned.rs:126-135).
inline svl_status widen_f32(const svl_tensor_view &t, int64_t numel, float *out) {
    if (t.dtype == SVL_F32) {
        const uint64_t expected = (uint64_t)numel * 4;
        if (t.nbytes != expected)
            return fail(SVL_CORRUPT, "tensor %s has %llu bytes, expected %llu for %lld F32 values",
                        t.name, (unsigned long long)t.nbytes, (unsigned long long)expected,
                        (long long)numel);
        if (numel > 0) std::memcpy(out, t.data, (size_t)numel * 4);
    } else if (t.dtype == SVL_BF16) {
        const uint64_t expected = (uint64_t)numel * 2;
        if (t.nbytes != expected)
            return fail(SVL_CORRUPT, "BF16 length mismatch: expected %llu bytes for %lld values, "
                        "got %llu", (unsigned long long)expected, (long long)numel,
                        (unsigned long long)t.nbytes);
        const uint16_t *b = (const uint16_t *)t.data;
        for (int64_t i = 0; i < numel; ++i) {
            const uint32_t bits = (uint32_t)b[i] << 16;
            std::memcpy(&out[(size_t)i], &bits, 4);
        }
    } else {
        return fail(SVL_UNSUPPORTED, "tensor %s has an unsupported dtype", t.name);
    }
    return SVL_OK;
}

inline svl_status decode_f32(const svl_tensor_view &t, int64_t numel, std::vector<float> &out) {
    out.resize((size_t)numel);
    if (svl_status st = widen_f32(t, numel, out.data())) return st;
    for (int64_t i = 0; i < numel; ++i)
        if (!std::isfinite(out[(size_t)i]))
            return fail(SVL_INTERNAL, "non-finite tensor value at index %lld of %s",
                        (long long)i, t.name);
    return SVL_OK;
}

inline svl_status decode_named(const TensorIndex &by_name, const std::string &name,
                               std::vector<float> &out) {
    auto it = by_name.find(name);
    if (it == by_name.end()) return fail(SVL_INTERNAL, "decoded tensor %s is missing", name.c_str());
    const svl_tensor_view *t = it->second;
    int64_t numel = 1;
    for (int d = 0; d < t->ndim; ++d) numel *= t->shape[d];
    return decode_f32(*t, numel, out);
}

// Copies a host array into a new device allocation recorded in `owned`.
inline svl_status upload_owned(std::vector<float *> &owned, const float *host, size_t count,
                               float **dst) {
    float *d = nullptr;
    HIP_TRY(hipMalloc((void **)&d, std::max<size_t>(count, 1) * sizeof(float)));
    owned.push_back(d);
    HIP_TRY(hipMemcpy(d, host, count * sizeof(float), hipMemcpyHostToDevice));
    *dst = d;
    return SVL_OK;
}

// The power of two that brings a bound on a split operand's magnitude into
// [2^13, 2^14) (halves reach 65504), within 2^-100 .. 2^100. From the bits: a
// model takes some 10^5 of them.
inline float split_scale(double bound) {
    if (!(bound > 0) || !std::isfinite(bound)) return 1.f;
    uint64_t b;
    std::memcpy(&b, &bound, sizeof b);
    const int e = (int)(b >> 52) - 1022;  // bound = f 2^e, f in [0.5, 1), but for denormals
    const uint32_t s = (uint32_t)(127 + std::max(-100, std::min(100, 14 - e))) << 23;
    float scale;
    std::memcpy(&scale, &s, sizeof scale);
    return scale;
}

// True where split_scale does bring it there (or there is nothing to bring).
inline bool split_scalable(double bound) {
    return bound == 0 || (bound >= 0x1p-80 && bound <= 0x1p80);
}

// One scale per channel of a split operand, from a bound on each channel's
// magnitude. A channel that stands out would otherwise set the scale of all,
// and the others' low halves would end in the half's denormals. The inverse
// scales go into the columns of the weight that reads the operand (0 for a
// channel that is always zero).
struct ChannelScales {
    std::vector<float> scale, inverse;
    bool ok = true;
    ChannelScales() = default;
    explicit ChannelScales(const std::vector<double> &bounds)
        : scale(bounds.size()), inverse(bounds.size()) {
        for (size_t i = 0; i < bounds.size(); ++i) {
            ok = ok && split_scalable(bounds[i]);
            scale[i] = split_scale(bounds[i]);
            inverse[i] = bounds[i] > 0 ? 1.f / scale[i] : 0.f;
        }
    }
};

// Largest magnitude of each channel of RMSNorm(x) * w: a normalised value is at
// most sqrt(n).
inline std::vector<double> norm_bounds(const std::vector<float> &w) {
    const double most = std::sqrt((double)w.size());
    std::vector<double> b(w.size());
    for (size_t i = 0; i < w.size(); ++i) b[i] = most * std::fabs((double)w[i]);
    return b;
}

template <class T>
inline double largest(const std::vector<T> &v) {
    double mx = 0;
    for (T x : v) mx = std::max(mx, (double)x);
    return mx;
}

// Query and key norm weights of a head, rotated in pairs (i, i + group / 2) of
// each `group` values: powers of two move between them so that both sides of a
// pair's products have like bounds (the products, and so the scores, stay the
// same numbers). False if the pairs' products still differ so much that more
// than a quarter would lose bits beside the largest (2^11 below it on each
// side, where a normalised value of 1 is scaled to about 2^-2).
inline bool balance_heads(std::vector<float> &qn, std::vector<float> &kn, size_t group) {
    std::vector<double> size;
    const size_t half = group / 2;
    for (size_t g = 0; g + group <= qn.size(); g += group)
        for (size_t i = g; i < g + half; ++i) {
            const float q = std::max(std::fabs(qn[i]), std::fabs(qn[i + half])),
                        k = std::max(std::fabs(kn[i]), std::fabs(kn[i + half]));
            if (q == 0.f || k == 0.f) {  // products of zero
                qn[i] = qn[i + half] = kn[i] = kn[i + half] = 0.f;
                continue;
            }
            if (!split_scalable(q) || !split_scalable(k)) return false;
            const int e = (std::ilogb(k) - std::ilogb(q)) >> 1;
            for (size_t j : {i, i + half}) {
                qn[j] = std::ldexp(qn[j], e);
                kn[j] = std::ldexp(kn[j], -e);
            }
            size.push_back(std::max(std::ldexp((double)q, e), std::ldexp((double)k, -e)));
        }
    const double least = std::ldexp(largest(size), -11);
    const int64_t small = std::count_if(size.begin(), size.end(), [&](double v) { return v < least; });
    return 4 * small <= (int64_t)size.size();
}

// Brings a model's projection weights to the device as split rows while the
// model is created (on the null stream; finish() waits). `fits` ends false when
// the halves would hold some operand in fewer bits than they should
// (split_rows_kernel and the bounds above say when): such a model is created
// again on FP32 operands.
struct SplitLoader {
    std::vector<float *> &owned;
    DevBuf<float> cols, mul;
    DevBuf<int> flag;
    bool fits = true;
    // The scale vectors' way to the device: pinned, so that a copy is only
    // enqueued (from pageable memory each waits, some 40 us; a tower takes 80).
    static constexpr size_t STAGE = (size_t)1 << 18;  // floats
    float *stage = nullptr;
    size_t staged = 0;

    explicit SplitLoader(std::vector<float *> &o) : owned(o) {}
    SplitLoader(const SplitLoader &) = delete;
    ~SplitLoader() {
        if (stage) {
            (void)hipStreamSynchronize(nullptr);
            (void)hipHostFree(stage);
        }
        cols.release();
        mul.release();
        flag.release();
    }

    svl_status put(DevBuf<float> &to, const std::vector<float> &v) {
        HIP_TRY(to.ensure(v.size()));
        if (v.size() > STAGE) {
            HIP_TRY(hipMemcpy(to.p, v.data(), v.size() * sizeof(float), hipMemcpyHostToDevice));
            return SVL_OK;
        }
        if (!stage)
            HIP_TRY(hipHostMalloc((void **)&stage, STAGE * sizeof(float), hipHostMallocDefault));
        if (staged + v.size() > STAGE) {
            HIP_TRY(hipStreamSynchronize(nullptr));  // the copies before have left it
            staged = 0;
        }
        std::copy(v.begin(), v.end(), stage + staged);
        HIP_TRY(hipMemcpyAsync(to.p, stage + staged, v.size() * sizeof(float),
                               hipMemcpyHostToDevice, nullptr));
        staged += v.size();
        return SVL_OK;
    }

    // A weight [rows, K] (K % 32 == 0), still FP32, with room for the descale
    // of each row behind it (K % 32 == 0 keeps it aligned).
    svl_status upload(const float *host, int64_t rows, int64_t K, float **w, float **wd) {
        const size_t count = (size_t)(rows * K);
        float *d = nullptr;
        HIP_TRY(hipMalloc((void **)&d, (count + (size_t)std::max<int64_t>(rows, 1)) * sizeof(float)));
        owned.push_back(d);
        HIP_TRY(hipMemcpy(d, host, count * sizeof(float), hipMemcpyHostToDevice));
        *w = d;
        *wd = d + count;
        return SVL_OK;
    }

    // Largest |RMSNorm(x) * norm . row| of each row of an uploaded FP32 weight
    // (Cauchy-Schwarz: sqrt(K) * |norm o row|; norm null: K-vectors of norm
    // sqrt(K)). `scratch`: rows floats on the device (the weight's descales).
    svl_status bounds(const float *w, int64_t rows, int64_t K, const std::vector<float> *norm,
                      float *scratch, std::vector<float> &each) {
        each.resize((size_t)rows);
        if (norm) ST_TRY(put(cols, *norm));
        HIP_TRY(launch_row_bounds(w, rows, (int)K, norm ? cols.p : nullptr, scratch, nullptr));
        HIP_TRY(hipMemcpy(each.data(), scratch, (size_t)rows * sizeof(float), hipMemcpyDeviceToHost));
        return SVL_OK;
    }

    // An uploaded weight to split rows in place, its columns times a's inverse
    // scales first (null: an A operand of one scale, a_scale); wd = the descale
    // of each output of its GEMM, times factor and row_mul[row].
    svl_status convert(float *w, int64_t rows, int64_t K, float a_scale, const ChannelScales *a,
                       float *wd, float factor = 1.f, const std::vector<float> *row_mul = nullptr) {
        if (!flag.p) {
            const int zero = 0;
            HIP_TRY(flag.ensure(1));
            HIP_TRY(hipMemcpy(flag.p, &zero, sizeof zero, hipMemcpyHostToDevice));
        }
        if (a) {
            fits = fits && a->ok;
            ST_TRY(put(cols, a->inverse));
        }
        if (row_mul) ST_TRY(put(mul, *row_mul));
        HIP_TRY(launch_split_rows(w, rows, (int)K, a ? cols.p : nullptr, factor / a_scale,
                                  row_mul ? mul.p : nullptr, wd, flag.p, nullptr));
        return SVL_OK;
    }

    svl_status weight(const std::vector<float> &host, int64_t K, float a_scale,
                      const ChannelScales *a, float **w, float **wd, float factor = 1.f) {
        const int64_t rows = (int64_t)host.size() / K;
        ST_TRY(upload(host.data(), rows, K, w, wd));
        return convert(*w, rows, K, a_scale, a, *wd, factor);
    }

    // A fused gate/up weight [2 I, K] (16-row blocks) over RMSNorm(x) * norm,
    // whose channels carry `in`: one scale per activation channel, |gelu(g) u|
    // being at most |g| |u|, applied by the up rows' descale.
    svl_status geglu(const std::vector<float> &gu, int64_t I, int64_t K,
                     const std::vector<float> &norm, const ChannelScales &in, float **w, float **wd,
                     ChannelScales &act) {
        std::vector<float> b;
        ST_TRY(upload(gu.data(), 2 * I, K, w, wd));
        ST_TRY(bounds(*w, 2 * I, K, &norm, *wd, b));
        auto at = [](int64_t j) { return (size_t)(32 * (j / 16) + j % 16); };
        std::vector<double> most((size_t)I);
        for (int64_t j = 0; j < I; ++j) {
            const double g = b[at(j)], u = b[at(j) + 16];
            fits = fits && split_scalable(g) && split_scalable(u);
            most[(size_t)j] = g * u;
        }
        act = ChannelScales(most);
        std::vector<float> row_mul((size_t)(2 * I), 1.f);
        for (int64_t j = 0; j < I; ++j) row_mul[at(j) + 16] = act.scale[(size_t)j];
        return convert(*w, 2 * I, K, 1.f, &in, *wd, 1.f, &row_mul);
    }

    svl_status finish(bool *ok) {
        int raised = 0;
        HIP_TRY(hipStreamSynchronize(nullptr));
        if (flag.p) HIP_TRY(hipMemcpy(&raised, flag.p, sizeof(int), hipMemcpyDeviceToHost));
        *ok = fits && raised == 0;
        return SVL_OK;
    }
};

// Gate and up projections [I, H] interleaved in blocks of `block` rows
// [g 0 .. block - 1, u 0 .. block - 1, g block .., ...], padded to I_pad rows
// each, for the GeGLU epilogue of the gate/up GEMM (32-row blocks for the
// FP32 GEMM, 16-row blocks for the split one).
inline std::vector<float> interleave_gate_up(const std::vector<float> &gate,
                                             const std::vector<float> &up, int64_t I,
                                             int64_t I_pad, int64_t H, int64_t block) {
    std::vector<float> gu((size_t)(2 * I_pad * H), 0.f);
    for (int64_t j = 0; j < I; ++j) {
        const int64_t at = 2 * block * (j / block) + j % block;
        std::copy(gate.begin() + j * H, gate.begin() + (j + 1) * H, gu.begin() + at * H);
        std::copy(up.begin() + j * H, up.begin() + (j + 1) * H, gu.begin() + (at + block) * H);
    }
    return gu;
}

// Device handle of a text model, for the image prompt glue: runs a text
// batch with soft-token features already in HBM (d_feats, rows indexed by
// featmap) and returns the normalized embeddings on the host.
svl_status text_forward_with_device_features(svl_text_model *m, const uint32_t *ids,
                                             const int64_t *offsets, int32_t batch,
                                             const int32_t *featmap, const float *d_feats,
                                             float *out_normalized);
int text_device(const svl_text_model *m);
int64_t text_hidden_size(const svl_text_model *m);
int64_t text_embedding_dim(const svl_text_model *m);
int64_t text_pad_token(const svl_text_model *m);

}  // namespace svl
