// PyTorch extension over the C ABI of libsbvr_hip.so: the operators that the
// reference binds in sbvr/kernels/sbvr_ops.cpp:152-172 (`_sbvr_mm_T`,
// `_sbvr_row_deq_mm_T`, `_sbvr_cuda_init`), with the same argument lists and the
// same shape inference from tensor sizes (:44-51, :90-96), plus the fp16
// activation linear over the default layout and its two one-row variants.
// This file holds no device code; it is the only C++ here that sees at::Tensor.
// Unlike the reference's wrappers it checks device, dtype and contiguity, guards
// the device and launches on torch's current HIP stream.  sbvr/hip.py offers the
// same operators through ctypes; both call the same entry points.
#include <torch/extension.h>

// (PyTorch on ROCm labels HIP devices "cuda"; these are the guard and stream types that accept that label)
#include <ATen/hip/HIPContext.h>
#include <ATen/hip/impl/HIPGuardImplMasqueradingAsCUDA.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <hip/hip_runtime_api.h>

#include <map>
#include <mutex>
#include <tuple>
#include <algorithm>
#include <stdexcept>
#include <string>
#include <vector>

#include "../../include/sbvr_hip.h"
#include "../../include/sbvr_hip_encoder.h"

namespace {

// Arguments that an operator does not take, as opposed to a device or an allocation that failed.
struct Refused : std::runtime_error {
    using std::runtime_error::runtime_error;
};

// The library reported an error of the device.
struct LaunchFailed : std::runtime_error {
    using std::runtime_error::runtime_error;
};

#define SBVR_WANT(cond, ...)                              \
    do {                                                  \
        if (!(cond))                                      \
            throw Refused(c10::str(__VA_ARGS__));         \
    } while (0)

using DeviceGuard = c10::hip::HIPGuardMasqueradingAsCUDA;

hipStream_t current_stream()
{
    return c10::hip::getCurrentHIPStreamMasqueradingAsCUDA().stream();
}

void want(const torch::Tensor &t, const char *name, c10::ScalarType dtype, int64_t dim, const torch::Tensor *like)
{
    SBVR_WANT(t.is_cuda(), name, " must be on a GPU (got ", t.device(), "); there is no CPU path");
    SBVR_WANT(t.scalar_type() == dtype, name, " must have dtype ", dtype, ", got ", t.scalar_type());
    SBVR_WANT(t.dim() == dim, name, " must have ", dim, " dimensions, got ", t.dim());
    SBVR_WANT(t.is_contiguous(), name, " must be contiguous");
    if (like)
        SBVR_WANT(t.device() == like->device(), name, " is on ", t.device(), ", expected ", like->device());
}

// uint8 indices for up to 256 lines, uint16 beyond (sbvr_kernel.cu:931-932)
int idx_bytes(const torch::Tensor &idx, int64_t lines, const char *name, const torch::Tensor &like)
{
    const auto expect = lines <= 256 ? torch::kUInt8 : torch::kUInt16;
    want(idx, name, expect, 2, &like);
    return lines <= 256 ? 1 : 2;
}

// the bias is used only when its length is N (sbvr_ops.cpp:56-58)
// (None is accepted beside the reference's 0-length tensor for "no bias")
using Bias = c10::optional<torch::Tensor>;

const void *bias_ptr(const Bias &bias, int64_t n, const torch::Tensor &like)
{
    if (!bias.has_value() || !bias->defined() || bias->numel() == 0 || bias->size(0) != n)
        return nullptr;
    want(*bias, "bias", torch::kFloat16, 1, &like);
    return bias->data_ptr();
}

void check(int rc)
{
    if (rc == SBVR_HIP_OK)
        return;
    const std::string message = c10::str("libsbvr_hip: error ", rc, ": ", sbvr_hip_last_error());
    if (rc == SBVR_HIP_ELAUNCH)
        throw LaunchFailed(message);
    throw Refused(message);
}

// (the entry points of sbvr_hip_encoder.h leave no message)
template <typename... Args>
void check_encoder(int rc, const char *what, const Args &...shape)
{
    if (rc == SBVR_HIP_OK)
        return;
    const std::string message = c10::str(what, ": error ", rc, shape...);
    if (rc == SBVR_HIP_ELAUNCH)
        throw LaunchFailed(message);
    throw Refused(message);
}

// Zero-initialised split-K accumulators per (device, stream), grown on demand to twice their size at least; the
// kernels leave the part that must be zero zeroed.  A buffer that is outgrown is kept until the process
// ends: a HIP graph captured earlier on that stream still holds its address (all of them together are smaller than
// the one in use).  One set for the linears of this file (SBVRLinear), one for the functions of sbvr/hip.py, whether
// they are launched here or through ctypes: a stream that one of these has warmed is warm for the others.  (Two sets,
// because the graphs of sbvr/decoder.py hold the second one's buffer of the stream they were recorded on and are
// replayed on others: a layer called on that stream meanwhile must not add into it.)
enum class Users { kLinears, kFunctions };

// While a graph is recorded on a stream whose buffer is missing or too small, the call gets one of the recording: its memory is
// the graph's, and the zeros are a node of the graph that has not run, so it is not kept for calls outside.  One per stream and
// set, dropped by the next such recording or the next buffer of its own.
torch::Tensor workspace(size_t nbytes, c10::Device device, hipStream_t stream, Users users)
{
    using Key = std::tuple<int, hipStream_t, Users>;
    static std::mutex mu;
    static std::map<Key, torch::Tensor> held;
    static std::map<Key, std::pair<unsigned long long, torch::Tensor>> recorded;       // (the recording's number, its buffer)
    static std::vector<torch::Tensor> outgrown;
    const Key key(static_cast<int>(device.index()), stream, users);
    auto enough = [&]() -> torch::Tensor {
        const auto it = held.find(key);
        return it != held.end() && static_cast<size_t>(it->second.numel()) >= nbytes ? it->second : torch::Tensor();
    };
    auto zeros = [&](size_t size) { return torch::zeros({static_cast<int64_t>(size)}, torch::dtype(torch::kUInt8).device(device)); };
    size_t size = std::max(nbytes, static_cast<size_t>(1) << 20);
    {
        std::lock_guard<std::mutex> lock(mu);
        torch::Tensor have = enough();
        if (have.defined())
            return have;
        if (held.count(key))
            size = std::max(size, 2 * static_cast<size_t>(held[key].numel()));
    }
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    unsigned long long recording = 0;
    if (hipStreamGetCaptureInfo(stream, &status, &recording) != hipSuccess) {
        status = hipStreamCaptureStatusNone;
        (void)hipGetLastError();             // (not the next launch's)
    }
    torch::Tensor made, dropped;             // (dropped: let go without the lock, as Python may hold the other end)
    if (status != hipStreamCaptureStatusNone) {
        {
            std::lock_guard<std::mutex> lock(mu);
            const auto it = recorded.find(key);
            if (it != recorded.end() && it->second.first == recording && static_cast<size_t>(it->second.second.numel()) >= nbytes)
                return it->second.second;
        }
        // (a smaller one of this recording: nodes recorded before keep its address, whose memory may serve nodes behind them)
        made = zeros(nbytes);
        std::lock_guard<std::mutex> lock(mu);
        auto &slot = recorded[key];
        dropped = std::move(slot.second);
        slot = {recording, made};
        return made;
    }
    // (allocated without the lock: torch may run Python on the way)
    made = zeros(size);
    std::lock_guard<std::mutex> lock(mu);
    torch::Tensor have = enough();           // (another thread on this stream was faster)
    if (have.defined())
        return have;
    if (held.count(key))
        outgrown.push_back(held[key]);
    const auto it = recorded.find(key);
    if (it != recorded.end()) {
        dropped = std::move(it->second.second);
        recorded.erase(it);
    }
    held[key] = made;
    return made;
}

// Elements per coefficient group: bvr_len where it is given, otherwise what `groups` rows of indices leave to each.
int64_t group_length(int64_t bvr_len, int64_t elements, int64_t groups, const char *name)
{
    SBVR_WANT(groups > 0, name, " has no groups");            // (an integer division by 0 would end the process)
    return bvr_len > 0 ? bvr_len : elements / groups;
}

struct LinearShape {
    int64_t M, N, K, S, G, L;
    int ib;
};

LinearShape linear_shape(int64_t M, int64_t K, const torch::Tensor &bvr, const torch::Tensor &coeff_idx,
                         const torch::Tensor &coeff_cache, int64_t bvr_len, const torch::Tensor &like)
{
    want(bvr, "bvr", torch::kUInt32, 3, &like);
    want(coeff_cache, "coeff_cache", torch::kFloat16, 2, &like);
    LinearShape s{};
    s.M = M;
    s.K = K;
    s.N = bvr.size(1);
    s.S = bvr.size(2);
    s.L = coeff_cache.size(0);
    s.ib = idx_bytes(coeff_idx, s.L, "coeff_idx", like);
    SBVR_WANT(bvr.size(0) * 32 == K, "x has K=", K, " but bvr holds ", bvr.size(0) * 32, " columns");
    SBVR_WANT(coeff_idx.size(1) == s.N && coeff_cache.size(1) == s.S, "coeff_idx / coeff_cache shapes do not match bvr");
    s.G = group_length(bvr_len, K, coeff_idx.size(0), "coeff_idx");
    SBVR_WANT(s.G * coeff_idx.size(0) == K, "coeff_idx has ", coeff_idx.size(0), " groups, K=", K, ", bvr_len=", s.G);
    return s;
}

}  // namespace

// Counterpart of sbvr_cuda_init (sbvr_ops.cpp:122-150): checks that the current device is a gfx950 part.
void sbvr_hip_init_current()
{
    check(sbvr_hip_init(static_cast<int>(at::hip::current_device())));
}

namespace {

// The launch of a linear over operands that have been checked; out: M * N elements.
void launch_linear(const torch::Tensor &x, const torch::Tensor &bvr, const torch::Tensor &coeff_idx, const torch::Tensor &coeff_cache,
                   const Bias &bias, const torch::Tensor &out, const LinearShape &s, int flags)
{
    hipStream_t stream = current_stream();
    // a prefill's partial results go to memory of the call's own (torch keeps it for the stream), which need not be cleared
    const size_t parts = sbvr_hip_linear_f16_parts(s.M, s.N, s.K, s.S, s.G);
    const size_t need = parts ? 0 : sbvr_hip_linear_f16_workspace(s.M, s.N, s.K, s.S, s.G);
    torch::Tensor ws = need ? workspace(need, x.device(), stream, Users::kLinears) : torch::Tensor();
    torch::Tensor scratch = parts ? at::empty({static_cast<int64_t>(parts)}, x.options().dtype(torch::kUInt8)) : torch::Tensor();
    check(sbvr_hip_linear_f16_scratch(x.data_ptr(), static_cast<const uint32_t *>(bvr.data_ptr()), coeff_idx.data_ptr(), s.ib,
                                      coeff_cache.data_ptr(), bias_ptr(bias, s.N, x), out.data_ptr(), s.M, s.N, s.K, s.S, s.G, s.L,
                                      need ? ws.data_ptr() : nullptr, need ? ws.numel() : 0, parts ? scratch.data_ptr() : nullptr, parts,
                                      flags, stream));
}

}  // namespace

// y = x @ decode(W)^T (+ bias): x (M, K) fp16; W in the default layout, bvr (K/32, N, S) uint32,
// coeff_idx (K/G, N), coeff_cache (L, S) fp16.  bvr_len <= 0: the group length follows from coeff_idx.
// out: an (M, N) fp16 tensor to write into (a caller that records a HIP graph brings its own), or None.
torch::Tensor sbvr_linear_f16(const torch::Tensor &x, const torch::Tensor &bvr, const torch::Tensor &coeff_idx,
                              const torch::Tensor &coeff_cache, const Bias &bias, int64_t bvr_len, int64_t flags,
                              const c10::optional<torch::Tensor> &out_opt)
{
    want(x, "x", torch::kFloat16, 2, nullptr);
    const LinearShape s = linear_shape(x.size(0), x.size(1), bvr, coeff_idx, coeff_cache, bvr_len, x);
    const DeviceGuard guard(x.device());
    torch::Tensor out;
    if (out_opt.has_value() && out_opt->defined()) {
        out = *out_opt;
        want(out, "out", torch::kFloat16, 2, &x);
        SBVR_WANT(out.size(0) == s.M && out.size(1) == s.N, "out has the wrong shape");
    } else {
        out = at::empty({s.M, s.N}, x.options());
    }
    launch_linear(x, bvr, coeff_idx, coeff_cache, bias, out, s, static_cast<int>(flags));
    return out;
}

// SBVRLinear.forward in one call: x (..., in_features) of any floating type; K zero-padded to k_padded where the encoder
// padded it, the output cut to out_features columns.  (Taking the steps of this one by one in Python cost as much
// as the launch: 9.2 us a call at 4096 -> 1024, one row, 5.0 to 5.4 in one.)
torch::Tensor sbvr_linear_forward(torch::Tensor x, const torch::Tensor &bvr, const torch::Tensor &coeff_idx,
                                  const torch::Tensor &coeff_cache, const Bias &bias, int64_t bvr_len, int64_t k_padded,
                                  int64_t out_features)
{
    SBVR_WANT(x.is_cuda(), "x must be on a GPU (got ", x.device(), "); there is no CPU path");
    SBVR_WANT(x.dim() >= 1, "x must have at least one dimension");
    SBVR_WANT(k_padded > 0, "the weight has no columns");
    if (x.scalar_type() != torch::kFloat16)
        x = x.to(torch::kFloat16);
    if (x.size(-1) != k_padded)
        x = at::constant_pad_nd(x, {0, k_padded - x.size(-1)});
    x = x.contiguous();
    const LinearShape s = linear_shape(x.numel() / k_padded, k_padded, bvr, coeff_idx, coeff_cache, bvr_len, x);
    const DeviceGuard guard(x.device());
    c10::SmallVector<int64_t, 6> sizes(x.sizes().begin(), x.sizes().end());
    sizes.back() = s.N;
    torch::Tensor out = at::empty(sizes, x.options());
    launch_linear(x, bvr, coeff_idx, coeff_cache, bias, out, s, 0);
    return s.N == out_features ? out : out.narrow(-1, 0, out_features);
}

// The linear of fp16(fp16(silu(gate)) * up) for gate_up (1, 2K) = gate | up.
torch::Tensor sbvr_linear_f16_swiglu(const torch::Tensor &gate_up, const torch::Tensor &bvr, const torch::Tensor &coeff_idx,
                                     const torch::Tensor &coeff_cache, const Bias &bias, int64_t bvr_len)
{
    want(gate_up, "gate_up", torch::kFloat16, 2, nullptr);
    SBVR_WANT(gate_up.size(1) % 2 == 0, "gate_up must have an even number of columns");
    const LinearShape s = linear_shape(gate_up.size(0), gate_up.size(1) / 2, bvr, coeff_idx, coeff_cache, bvr_len, gate_up);
    const DeviceGuard guard(gate_up.device());
    hipStream_t stream = current_stream();
    auto out = torch::empty({s.M, s.N}, torch::dtype(torch::kFloat16).device(gate_up.device()));
    const size_t need = sbvr_hip_linear_f16_workspace(s.M, s.N, s.K, s.S, s.G);
    torch::Tensor ws = need ? workspace(need, gate_up.device(), stream, Users::kLinears) : torch::Tensor();
    check(sbvr_hip_linear_f16_swiglu(gate_up.data_ptr(), static_cast<const uint32_t *>(bvr.data_ptr()), coeff_idx.data_ptr(),
                                     s.ib, coeff_cache.data_ptr(), bias_ptr(bias, s.N, gate_up), out.data_ptr(), s.M, s.N,
                                     s.K, s.S, s.G, s.L, need ? ws.data_ptr() : nullptr, need ? ws.numel() : 0, stream));
    return out;
}

// x_out <- r = fp16(x + delta); returns the linear of norm_weight * fp16(r * rsqrt(mean(r^2) + eps)).
torch::Tensor sbvr_linear_f16_add_rmsnorm(torch::Tensor x, torch::Tensor delta, torch::Tensor norm_weight, double eps,
                                          torch::Tensor x_out, torch::Tensor bvr, torch::Tensor coeff_idx,
                                          torch::Tensor coeff_cache, Bias bias, int64_t bvr_len)
{
    want(x, "x", torch::kFloat16, 2, nullptr);
    want(delta, "delta", torch::kFloat16, 2, &x);
    want(x_out, "x_out", torch::kFloat16, 2, &x);
    want(norm_weight, "norm_weight", torch::kFloat16, 1, &x);
    SBVR_WANT(x.size(0) == 1 && delta.sizes() == x.sizes() && x_out.sizes() == x.sizes() &&
                    norm_weight.size(0) == x.size(1),
                "x, delta and x_out must be (1, K) and norm_weight (K)");
    const LinearShape s = linear_shape(1, x.size(1), bvr, coeff_idx, coeff_cache, bvr_len, x);
    const DeviceGuard guard(x.device());
    hipStream_t stream = current_stream();
    auto out = torch::empty({1, s.N}, torch::dtype(torch::kFloat16).device(x.device()));
    const size_t need = sbvr_hip_linear_f16_workspace(1, s.N, s.K, s.S, s.G);
    torch::Tensor ws = need ? workspace(need, x.device(), stream, Users::kLinears) : torch::Tensor();
    check(sbvr_hip_linear_f16_add_rmsnorm(x.data_ptr(), delta.data_ptr(), norm_weight.data_ptr(), static_cast<float>(eps),
                                          x_out.data_ptr(), static_cast<const uint32_t *>(bvr.data_ptr()),
                                          coeff_idx.data_ptr(), s.ib, coeff_cache.data_ptr(), bias_ptr(bias, s.N, x),
                                          out.data_ptr(), s.N, s.K, s.S, s.G, s.L, need ? ws.data_ptr() : nullptr,
                                          need ? ws.numel() : 0, stream));
    return out;
}

// Both operands encoded, default layout: l_bvr (K/32, M, Sl), r_bvr (K/32, N, Sr) (sbvr_ops.cpp:35-76).
// bvr_len <= 0: the group length follows from l_coeff_idx.
torch::Tensor sbvr_mm_T(const torch::Tensor &l_bvr, const torch::Tensor &l_coeff_idx, const torch::Tensor &l_coeff_cache,
                        const torch::Tensor &r_bvr, const torch::Tensor &r_coeff_idx, const torch::Tensor &r_coeff_cache,
                        const Bias &bias, int64_t bvr_len)
{
    want(l_bvr, "l_bvr", torch::kUInt32, 3, nullptr);
    want(r_bvr, "r_bvr", torch::kUInt32, 3, &l_bvr);
    want(l_coeff_cache, "l_coeff_cache", torch::kFloat16, 2, &l_bvr);
    want(r_coeff_cache, "r_coeff_cache", torch::kFloat16, 2, &l_bvr);
    const int64_t M = l_bvr.size(1), N = r_bvr.size(1), K = l_bvr.size(0) * 32;
    const int64_t Sl = l_bvr.size(2), Sr = r_bvr.size(2), Ll = l_coeff_cache.size(0), Lr = r_coeff_cache.size(0);
    SBVR_WANT(l_bvr.size(0) == r_bvr.size(0), "operands disagree on K: ", K, " vs ", r_bvr.size(0) * 32);
    const int lib = idx_bytes(l_coeff_idx, Ll, "l_coeff_idx", l_bvr), rib = idx_bytes(r_coeff_idx, Lr, "r_coeff_idx", l_bvr);
    SBVR_WANT(l_coeff_idx.size(1) == M && r_coeff_idx.size(1) == N && l_coeff_idx.size(0) == r_coeff_idx.size(0) &&
                    l_coeff_cache.size(1) == Sl && r_coeff_cache.size(1) == Sr,
                "index / table shapes do not match the bit planes");
    const int64_t G = group_length(bvr_len, K, l_coeff_idx.size(0), "l_coeff_idx");
    SBVR_WANT(G * l_coeff_idx.size(0) == K, "coeff_idx has ", l_coeff_idx.size(0), " groups, K=", K);
    const DeviceGuard guard(l_bvr.device());
    auto out = at::empty({M, N}, l_coeff_cache.options());
    hipStream_t stream = current_stream();
    const size_t need = sbvr_hip_mm_T_workspace(static_cast<int>(M), static_cast<int>(N));
    torch::Tensor ws;                    // (no split of K for this call: no workspace, nothing allocated)
    if (need)
        ws = workspace(need, l_bvr.device(), stream, Users::kFunctions);
    check(sbvr_hip_mm_T_ws(static_cast<const uint32_t *>(l_bvr.data_ptr()), l_coeff_idx.data_ptr(), lib,
                           l_coeff_cache.data_ptr(), static_cast<const uint32_t *>(r_bvr.data_ptr()), r_coeff_idx.data_ptr(),
                           rib, r_coeff_cache.data_ptr(), bias_ptr(bias, N, l_bvr), out.data_ptr(), M, N, K, Sl, Sr, G, Ll,
                           Lr, need ? ws.data_ptr() : nullptr, need, stream));
    return out;
}

// Activations x (M, K) fp16 encoded against one line of input coefficients per group of K, lines (K/G, S) fp16: the
// left operand's (bvr, coeff_idx) (what sbvr/core.py:1021-1022 of the reference is a placeholder for).
std::tuple<torch::Tensor, torch::Tensor> sbvr_online_encode_lines(const torch::Tensor &x, const torch::Tensor &lines, int64_t bvr_len)
{
    want(x, "x", torch::kFloat16, 2, nullptr);
    want(lines, "lines", torch::kFloat16, 2, &x);
    const int64_t M = x.size(0), K = x.size(1), groups = lines.size(0), S = lines.size(1);
    SBVR_WANT(K == groups * bvr_len, "lines must be (K / bvr_len, S), got ", lines.sizes(), " for K=", K, ", bvr_len=", bvr_len);
    const DeviceGuard guard(x.device());
    auto bvr = at::empty({K / 32, M, S}, x.options().dtype(torch::kUInt32));
    auto idx = at::empty({groups, M}, x.options().dtype(groups <= 256 ? torch::kUInt8 : torch::kUInt16));
    const int rc = sbvr_hip_online_encode_lines_f16(x.data_ptr(), lines.data_ptr(), static_cast<uint32_t *>(bvr.data_ptr()), idx.data_ptr(),
                                                    groups <= 256 ? 1 : 2, M, K, bvr_len, S, current_stream());
    check_encoder(rc, "sbvr_hip_online_encode_lines_f16", " (M=", M, " K=", K, " bvr_len=", bvr_len, " S=", S, ")");
    return {bvr, idx};
}

// sbvr.online_mm_T in one call: x (..., K) activations of any floating type, K zero-padded to the groups of `lines`, encoded
// against them and multiplied with the encoded weight.  (Step by step from Python a call took 20 us, 12 of them the host's.)
torch::Tensor sbvr_online_mm_T(torch::Tensor x, const torch::Tensor &lines, const torch::Tensor &r_bvr, const torch::Tensor &r_coeff_idx,
                               const torch::Tensor &r_coeff_cache, const Bias &bias, int64_t bvr_len)
{
    const c10::InferenceMode inference;             // (what the method it serves runs under)
    SBVR_WANT(x.is_cuda() && x.device() == r_bvr.device(), "x must be on the weight's GPU");
    SBVR_WANT(lines.dim() == 2 && bvr_len > 0, "lines must be (K / bvr_len, S)");
    const int64_t K = lines.size(0) * bvr_len;
    SBVR_WANT(x.dim() >= 1 && x.size(-1) > 0 && x.size(-1) <= K && K - x.size(-1) < bvr_len, "x does not fit the input coefficients");
    if (x.dim() != 2)
        x = x.reshape({-1, x.size(-1)});
    if (x.scalar_type() != torch::kFloat16)
        x = x.to(torch::kFloat16);
    if (x.size(1) != K)
        x = at::constant_pad_nd(x, {0, K - x.size(1)});
    const torch::Tensor table = lines.contiguous();
    if (x.size(0) > 0 && table.scalar_type() == torch::kFloat16 && table.device() == x.device() && r_bvr.dim() == 3 && r_bvr.scalar_type() == torch::kUInt32 &&
        r_bvr.is_contiguous() && r_bvr.size(0) * 32 == K && r_coeff_cache.dim() == 2) {
        const int64_t M = x.size(0), N = r_bvr.size(1), Sl = table.size(1), Sr = r_bvr.size(2), Lr = r_coeff_cache.size(0);
        const size_t need = M < (1 << 20) && K < (1 << 30) ? sbvr_hip_online_mm_T_scratch(static_cast<const uint32_t *>(r_bvr.data_ptr()), r_coeff_cache.data_ptr(),
                                                                                         M, N, K, Sl, Sr, bvr_len) : 0;
        if (need) {
            want(r_coeff_cache, "r_coeff_cache", torch::kFloat16, 2, &x);
            const int rib = idx_bytes(r_coeff_idx, Lr, "r_coeff_idx", x);
            SBVR_WANT(r_coeff_idx.size(1) == N && r_coeff_idx.size(0) * bvr_len == K && r_coeff_cache.size(1) == Sr,
                      "index / table shapes do not match the bit planes");
            const DeviceGuard guard(x.device());
            const torch::Tensor xc = x.contiguous();
            auto out = at::empty({M, N}, table.options());
            auto scratch = at::empty({static_cast<int64_t>(need)}, table.options().dtype(torch::kUInt8));
            const int rc = sbvr_hip_online_mm_T(xc.data_ptr(), table.data_ptr(), static_cast<const uint32_t *>(r_bvr.data_ptr()), r_coeff_idx.data_ptr(), rib,
                                                r_coeff_cache.data_ptr(), bias_ptr(bias, N, x), out.data_ptr(), M, N, K, Sl, Sr, bvr_len, Lr,
                                                scratch.data_ptr(), need, current_stream());
            check_encoder(rc, "sbvr_hip_online_mm_T", " (M=", M, " N=", N, " K=", K, " bvr_len=", bvr_len, " S=", Sl, ",", Sr, ")");
            return out;
        }
    }
    const auto [bvr, idx] = sbvr_online_encode_lines(x.contiguous(), table, bvr_len);
    return sbvr_mm_T(bvr, idx, table, r_bvr, r_coeff_idx, r_coeff_cache, bias, 0);
}

// The dense (N, cols) weight of a default-layout encoding, fp16, bf16 or fp32 (sbvr/core.py:926-949).
torch::Tensor sbvr_decode_weight(const torch::Tensor &bvr, const torch::Tensor &coeff_idx, const torch::Tensor &coeff_cache,
                                 int64_t bvr_len, int64_t cols, c10::ScalarType dtype)
{
    want(bvr, "bvr", torch::kUInt32, 3, nullptr);
    want(coeff_cache, "coeff_cache", torch::kFloat16, 2, &bvr);
    SBVR_WANT(coeff_idx.scalar_type() == torch::kUInt8 || coeff_idx.scalar_type() == torch::kUInt16, "coeff_idx must be uint8 or uint16");
    want(coeff_idx, "coeff_idx", coeff_idx.scalar_type(), 2, &bvr);
    const int64_t K = bvr.size(0) * 32, N = bvr.size(1), S = bvr.size(2), L = coeff_cache.size(0);
    SBVR_WANT(coeff_idx.size(0) * bvr_len == K && coeff_idx.size(1) == N && coeff_cache.size(1) == S,
                "coeff_idx / coeff_cache shapes do not match bvr");
    const int type = dtype == torch::kFloat32 ? 2 : (dtype == torch::kBFloat16 ? 1 : 0);
    const DeviceGuard guard(bvr.device());
    auto out = at::empty({N, cols}, coeff_cache.options().dtype(type == 2 ? torch::kFloat32 : (type == 1 ? torch::kBFloat16 : torch::kFloat16)));
    const int rc = sbvr_hip_decode_weight(static_cast<const uint32_t *>(bvr.data_ptr()), coeff_idx.data_ptr(),
                                          static_cast<int>(coeff_idx.element_size()), coeff_cache.data_ptr(), out.data_ptr(), type, N, K,
                                          cols, S, bvr_len, L, current_stream());
    check_encoder(rc, "sbvr_hip_decode_weight", " (N=", N, " K=", K, " cols=", cols, " S=", S, " bvr_len=", bvr_len, ")");
    return out.scalar_type() == dtype ? out : out.to(dtype);
}

// The same under the inference mode of sbvr.decode.
torch::Tensor sbvr_decode(const torch::Tensor &bvr, const torch::Tensor &coeff_idx, const torch::Tensor &coeff_cache, int64_t bvr_len,
                          int64_t cols, c10::ScalarType dtype)
{
    const c10::InferenceMode inference;
    return sbvr_decode_weight(bvr, coeff_idx, coeff_cache, bvr_len, cols, dtype);
}

// fp16 l_w (M, K) against a trans=True weight: r_bvr (N/32, K, S), r_coeff_idx (N/G, K) (sbvr_ops.cpp:79-120).
// use_shfl chose between equivalent CUDA kernels in the reference and is ignored.
// bvr_len <= 0: the group length follows from r_coeff_idx.
torch::Tensor sbvr_row_deq_mm_T(const torch::Tensor &l_w, const torch::Tensor &r_bvr, const torch::Tensor &r_coeff_idx,
                                const torch::Tensor &r_coeff_cache, const Bias &bias, int64_t use_shfl, int64_t bvr_len)
{
    (void)use_shfl;
    want(l_w, "l_w", torch::kFloat16, 2, nullptr);
    want(r_bvr, "r_bvr", torch::kUInt32, 3, &l_w);
    want(r_coeff_cache, "r_coeff_cache", torch::kFloat16, 2, &l_w);
    const int64_t M = l_w.size(0), K = l_w.size(1), N = r_bvr.size(0) * 32, S = r_bvr.size(2), L = r_coeff_cache.size(0);
    const int ib = idx_bytes(r_coeff_idx, L, "r_coeff_idx", l_w);
    SBVR_WANT(r_bvr.size(1) == K && r_coeff_idx.size(1) == K && r_coeff_cache.size(1) == S, "operand shapes do not match");
    const int64_t G = group_length(bvr_len, N, r_coeff_idx.size(0), "r_coeff_idx");
    SBVR_WANT(G * r_coeff_idx.size(0) == N, "r_coeff_idx has ", r_coeff_idx.size(0), " groups, N=", N);
    const DeviceGuard guard(l_w.device());
    auto out = at::empty({M, N}, l_w.options());
    hipStream_t stream = current_stream();
    const size_t need = sbvr_hip_row_deq_mm_T_workspace_for(static_cast<int>(M), static_cast<int>(N), static_cast<int>(K),
                                                            static_cast<int>(S), static_cast<int>(G));
    torch::Tensor ws;                    // (no split of K for this call: no workspace, nothing allocated)
    if (need)
        ws = workspace(need, l_w.device(), stream, Users::kFunctions);
    check(sbvr_hip_row_deq_mm_T_ws(l_w.data_ptr(), static_cast<const uint32_t *>(r_bvr.data_ptr()), r_coeff_idx.data_ptr(), ib,
                                   r_coeff_cache.data_ptr(), bias_ptr(bias, N, l_w), out.data_ptr(), M, N, K, S, G, L,
                                   need ? ws.data_ptr() : nullptr, need, stream));
    return out;
}

// The functions' workspace of the current stream of a device, for launches that are made through the C ABI.
torch::Tensor workspace_of_current_stream(int64_t nbytes, int64_t device)
{
    const c10::Device dev(c10::DeviceType::CUDA, static_cast<c10::DeviceIndex>(device));
    const DeviceGuard guard(dev);
    return workspace(static_cast<size_t>(nbytes), dev, current_stream(), Users::kFunctions);
}

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m)
{
    namespace py = pybind11;
    py::register_exception<Refused>(m, "Refused", PyExc_RuntimeError);
    py::register_exception<LaunchFailed>(m, "LaunchFailed", PyExc_RuntimeError);
    // (the operators that sbvr/hip.py calls: other Python threads run on while a launch waits for room in its queue)
    const py::call_guard<py::gil_scoped_release> no_gil;
    m.def("_sbvr_hip_init", &sbvr_hip_init_current, "Checks that the current device is a gfx950 part");
    m.def("_sbvr_cuda_init", &sbvr_hip_init_current, "Alias of _sbvr_hip_init under the reference's name");
    m.def("_sbvr_mm_T", &sbvr_mm_T, "SBVR x SBVR^T, both operands encoded", py::arg("l_bvr"), py::arg("l_coeff_idx"),
          py::arg("l_coeff_cache"), py::arg("r_bvr"), py::arg("r_coeff_idx"), py::arg("r_coeff_cache"), py::arg("bias"),
          py::arg("bvr_len") = 0, no_gil);
    m.def("_sbvr_row_deq_mm_T", &sbvr_row_deq_mm_T, "fp16 x SBVR^T over the trans=True layout", py::arg("l_w"),
          py::arg("r_bvr"), py::arg("r_coeff_idx"), py::arg("r_coeff_cache"), py::arg("bias"), py::arg("use_shfl") = 0,
          py::arg("bvr_len") = 0, no_gil);
    m.def("_sbvr_linear_f16", &sbvr_linear_f16, "fp16 x SBVR^T over the default layout", py::arg("x"), py::arg("bvr"),
          py::arg("coeff_idx"), py::arg("coeff_cache"), py::arg("bias") = py::none(), py::arg("bvr_len") = 0,
          py::arg("flags") = 0, py::arg("out") = py::none());
    m.def("_linear_forward", &sbvr_linear_forward, "SBVRLinear.forward", py::arg("x"), py::arg("bvr"), py::arg("coeff_idx"),
          py::arg("coeff_cache"), py::arg("bias"), py::arg("bvr_len"), py::arg("k_padded"), py::arg("out_features"));
    m.def("_online_encode_lines", &sbvr_online_encode_lines, "activations to the arrays of an encoded left operand", py::arg("x"),
          py::arg("lines"), py::arg("bvr_len"), no_gil);
    m.def("_online_mm_T", &sbvr_online_mm_T, "sbvr.online_mm_T", py::arg("x"), py::arg("lines"), py::arg("r_bvr"), py::arg("r_coeff_idx"),
          py::arg("r_coeff_cache"), py::arg("bias"), py::arg("bvr_len"), no_gil);
    m.def("_decode_weight", &sbvr_decode_weight, "the dense weight of a default-layout encoding", py::arg("bvr"),
          py::arg("coeff_idx"), py::arg("coeff_cache"), py::arg("bvr_len"), py::arg("cols"), py::arg("dtype"), no_gil);
    m.def("_decode", &sbvr_decode, "sbvr.decode", py::arg("bvr"), py::arg("coeff_idx"), py::arg("coeff_cache"), py::arg("bvr_len"),
          py::arg("cols"), py::arg("dtype"), no_gil);
    m.def("_workspace", &workspace_of_current_stream, "the split-K workspace of the device's current stream", py::arg("nbytes"),
          py::arg("device"));
    m.def("last_kernel", &sbvr_hip_last_kernel, "which kernel the last linear call of this thread launched");
    m.def("_sbvr_linear_f16_swiglu", &sbvr_linear_f16_swiglu, "the linear of silu(gate) * up, one row", py::arg("gate_up"),
          py::arg("bvr"), py::arg("coeff_idx"), py::arg("coeff_cache"), py::arg("bias") = py::none(),
          py::arg("bvr_len") = 0);
    m.def("_sbvr_linear_f16_add_rmsnorm", &sbvr_linear_f16_add_rmsnorm, "x_out <- x + delta, the linear of its RMSNorm",
          py::arg("x"), py::arg("delta"), py::arg("norm_weight"), py::arg("eps"), py::arg("x_out"), py::arg("bvr"),
          py::arg("coeff_idx"), py::arg("coeff_cache"), py::arg("bias") = py::none(), py::arg("bvr_len") = 0);
    m.def("version", &sbvr_hip_version, "ABI version of the library underneath");
}
