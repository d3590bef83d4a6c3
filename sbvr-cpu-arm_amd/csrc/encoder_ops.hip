// Encoder search on the GPU (libsbvr_hip.so, gfx950): the error of every (group, candidate line) pair of
// the SBVR encoder's search, for many groups at once.
//
// The search (reference sbvr/core.py:485-501, _data_diff_min_mse) takes a group of G values and n candidate
// lines, each line given by its 2^S subset sums ("points"), and wants, per line, the mean over the group of
// the squared distance from each value to its nearest point.  The reference forms the (n, G, 2^S) tensor of
// squared differences in the compute type and reduces it; at 4096 x 4096 that tensor is written and read
// 131072 times.  Here a thread owns one (group, line) pair, keeps the line's points in registers and walks
// the group's values (in LDS, read as broadcasts): nothing but the (groups, lines) matrix of errors goes to
// memory.  The arithmetic per element is the reference's: fp16 subtraction, fp16 square, minimum (packed,
// two points per instruction), then an fp32 sum over the group in element order and one division.

#include "../../include/sbvr_hip_encoder.h"
#include "sbvr_internal.h"
#include "sbvr_device.h"

namespace {

constexpr int kEncThreads = 256;
constexpr int kEncMaxG = 4096;        // values of a group the LDS copy holds at a time (8 KiB)

// P points per line (a power of two, 2 <= P <= 256).  Grid: (ceil(n / 256), groups).  Groups longer than the
// LDS copy go through it in pieces.
template <int P>
__global__ void __launch_bounds__(kEncThreads)
sbvr_encoder_group_mse_kernel(const uint16_t *__restrict__ data, const uint16_t *__restrict__ points,
                              float *__restrict__ mse, int G, int n)
{
    __shared__ __align__(16) uint16_t group[kEncMaxG];
    const int b = blockIdx.y;
    const uint16_t *mine = data + static_cast<size_t>(b) * G;
    const int line = blockIdx.x * kEncThreads + threadIdx.x;
    const int line_c = min(line, n - 1);          // (threads past the end repeat the last line and store nothing)
    v2h p[P / 2];
    const uint32_t *src = reinterpret_cast<const uint32_t *>(points + static_cast<size_t>(line_c) * P);
#pragma unroll
    for (int j = 0; j < P / 2; ++j)
        p[j] = __builtin_bit_cast(v2h, src[j]);

    float sum = 0.f;
    for (int g0 = 0; g0 < G; g0 += kEncMaxG) {
        const int len = min(G - g0, kEncMaxG);
        __syncthreads();
        for (int i = threadIdx.x; i < len; i += kEncThreads)
            group[i] = mine[g0 + i];
        __syncthreads();
        for (int g = 0; g < len; ++g) {
            const uint16_t raw = group[g];
            const _Float16 d = __builtin_bit_cast(_Float16, raw);
            const v2h dd = {d, d};
            v2h best;
#pragma unroll
            for (int j = 0; j < P / 2; ++j) {
                const v2h diff = dd - p[j];
                const v2h sq = diff * diff;
                best = j == 0 ? sq : __builtin_elementwise_min(best, sq);
            }
            const _Float16 m = best[0] < best[1] ? best[0] : best[1];
            sum += static_cast<float>(m);
        }
    }
    if (line < n)
        mse[static_cast<size_t>(b) * n + line] = sum / static_cast<float>(G);
}

// The candidate lines of one group's search, formed and measured in one launch: first the geometric families
// b + s * base (reference sbvr/core.py:392-403; index (b, s, base), the last fastest; fp16 product, fp16 sum), then the
// grid of S axes of `steps` values each (core.py:368-390; the last axis fastest).  A thread owns a candidate: its
// coefficients go to `lines` as they are formed (the winner's are read back), its 2^S subset sums (fp32 sums rounded
// to fp16 once) stay in registers, and its error follows as in the kernel above.  The order of a line's coefficients
// does not change its points, so only the winner has to be sorted.  Bound by the vector ALU: three packed operations
// per two points and value.  (Formed by torch, 2.6e5 to 4.6e5 lines of 4 coefficients were written, concatenated,
// sorted, gathered and multiplied out to points before the kernel above read them: a 1024 x 4096 weight with groups of
// 128 took 424-454 ms to encode, 294-307 ms with this launch.)
struct CandidateArgs {
    const uint16_t *data, *base, *b, *s, *axes;
    uint16_t *lines;
    float *mse;
    int bases, ss, steps, family, n, G;
};

template <int S>
__global__ void __launch_bounds__(kEncThreads)
sbvr_encoder_candidates_kernel(const CandidateArgs a)
{
#pragma clang fp contract(off)
    constexpr int P = 1 << S;
    __shared__ __align__(16) uint16_t group[kEncMaxG];
    for (int i = threadIdx.x; i < a.G; i += kEncThreads)
        group[i] = a.data[i];
    __syncthreads();
    const int line = blockIdx.x * kEncThreads + threadIdx.x;
    const int at = min(line, a.n - 1);
    auto half_of = [](uint16_t v) __attribute__((always_inline)) -> _Float16 { return __builtin_bit_cast(_Float16, v); };
    _Float16 c[S];
    if (at < a.family) {
        const int ir = at % a.bases, is = at / a.bases % a.ss, ib = at / a.bases / a.ss;
        const _Float16 sv = half_of(a.s[is]), bv = half_of(a.b[ib]);
#pragma unroll
        for (int q = 0; q < S; ++q) {
            const _Float16 scaled = sv * half_of(a.base[ir * S + q]);
            c[q] = bv + scaled;
        }
    } else {
        int rest = at - a.family;
#pragma unroll
        for (int q = S - 1; q >= 0; --q) {
            c[q] = half_of(a.axes[q * a.steps + rest % a.steps]);
            rest /= a.steps;
        }
    }
    float sums[P];
    sums[0] = 0.f;
#pragma unroll
    for (int q = 0; q < S; ++q)
#pragma unroll
        for (int i = 0; i < (1 << q); ++i)
            sums[(1 << q) + i] = sums[i] + static_cast<float>(c[q]);
    v2h p[P / 2];
#pragma unroll
    for (int j = 0; j < P / 2; ++j)
        p[j] = v2h{static_cast<_Float16>(sums[2 * j]), static_cast<_Float16>(sums[2 * j + 1])};

    float sum = 0.f;
    for (int g = 0; g < a.G; g += 4) {                        // (G is a multiple of 4)
        const uint2 four = *reinterpret_cast<const uint2 *>(group + g);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const uint32_t pair = e < 2 ? four.x : four.y;
            const _Float16 d = half_of(static_cast<uint16_t>(e & 1 ? pair >> 16 : pair));
            const v2h dd = {d, d};
            v2h best;
#pragma unroll
            for (int j = 0; j < P / 2; ++j) {
                const v2h diff = dd - p[j];
                const v2h sq = diff * diff;
                best = j == 0 ? sq : __builtin_elementwise_min(best, sq);
            }
            const _Float16 m = best[0] < best[1] ? best[0] : best[1];
            sum += static_cast<float>(m);
        }
    }
    if (line < a.n) {
#pragma unroll
        for (int q = 0; q < S; ++q)
            a.lines[static_cast<size_t>(line) * S + q] = __builtin_bit_cast(uint16_t, c[q]);
        a.mse[line] = sum / static_cast<float>(a.G);
    }
}

// ------------------------------------------------------------------- the search of new lines, group after group
//
// The encoder's policy is a chain: a group that the table does not serve (its best error is not below the cut-off)
// searches the candidate lines, the line it finds may join the table and moves the cut-off, and both decide what the
// groups behind it find (sbvr/core.py:555-653).  Here the chain runs on the device: every group carries its best error
// over the table (best, line), and a round of two launches takes the next group that misses through its search,
//   search:  the bounds and axes of its candidates, worked out by every workgroup for itself, then a candidate a thread;
//   settle:  the winner joins the table or not, the cut-off moves, every group behind it meets the new line, and the
//            first of those that now misses is the next round's (an atomic minimum).
// The host queues rounds ahead and looks at the state now and then; rounds behind the last miss do nothing, and so do
// those behind a group whose candidates these kernels do not form (status 1: the host takes that group through
// the general path).  State: two slots, read one and written the other by turns, so that workgroups of a launch never
// read what it changes, but for `found` of the slot read, which the search takes minima into (and reads as a bound).  That a group
// is left to the host the search says in the other slot, for the settling launch: its group is this one already, where otherwise
// it is one behind.
// A workgroup's search is bound by the vector ALU (3 packed operations per two points and value); a wave stops when
// all of its 64 lines are above the best error known.  1024 x 4096, groups of 128, 4 planes (241 misses): 269 to 327 ms
// with about 50 launches and two waits a miss, 9.6 to 10.9 here: 22 us a search (2.6e5 to 4.6e5 lines; 38 to 59 without
// the bound), 8 to settle it (windows of 2048 groups meet the table as their turn comes near; 23 with all of up to 32768 groups
// behind a miss meeting every line).
struct EncoderState {
    int lines, misses, history, status, miss;
    int unmet;                           // groups at the end that have not met the table; those in front have met all of its lines
    unsigned long long found;            // error's bits << 32 | candidate: the least so far (all ones: none)
};

constexpr int kEncMaxScales = 160, kEncMaxAxes = 4096;    // scales of a search, values of all its axes, at most
constexpr int kEncSettleValues = 1024;                    // squared distances of a workgroup's groups in LDS (of one, where it is longer)
constexpr int kEncWindow = 2048;                          // groups that meet the table in one go
constexpr int kEncNone = 0x7fffffff;

// torch.linspace in fp16: the step rounded, values from either end.
__device__ __forceinline__ _Float16 line_space(_Float16 lo, _Float16 hi, int n, int i)
{
#pragma clang fp contract(off)
    const _Float16 span = hi - lo;
    const _Float16 step = static_cast<_Float16>(static_cast<float>(span) / static_cast<float>(static_cast<_Float16>(static_cast<float>(n - 1))));
    const float s = static_cast<float>(step);
    return i < n / 2 ? fma_half(s, static_cast<float>(i), static_cast<float>(lo))
                     : fma_half(-s, static_cast<float>(n - 1 - i), static_cast<float>(hi));
}

// The scales of a group's search (GroupEncoder.candidate_lines): from, from + step, ...
struct Scales {
    float from, step;
    double count;
    int wide;
};

__device__ __forceinline__ Scales search_scales(const sbvr_hip_encoder_run &a, const EncoderState &st, float q95, _Float16 hl, _Float16 hh)
{
#pragma clang fp contract(off)
    Scales r;
    // hits so far over groups so far, this one counted: above 0.6 (and while the table fills) the wider search
    const double seen = static_cast<double>(a.before) + st.miss;
    r.wide = st.lines < a.warmup || (seen - st.misses) / (seen + 1.) > 0.6;
    const _Float16 s_hi = fma_half(static_cast<float>(static_cast<_Float16>(hh - hl)), 1.1f, 0.f);
    const float s_lo = 2.f * q95;
    r.step = (static_cast<float>(s_hi) - s_lo) * a.scale_step;
    if (r.wide)
        r.step = r.step * a.scale_narrow;
    r.from = s_lo + r.step;
    const float to = static_cast<float>(s_hi) + r.step;
    r.count = ceil((static_cast<double>(to) - static_cast<double>(r.from)) / static_cast<double>(r.step));
    if (!(fabsf(to) < INFINITY))
        r.count = 0.;
    return r;
}

// Value i of axis q: from a margin below the data's edge q to one above edge q + 1.
template <int S>
__device__ __forceinline__ _Float16 axis_value(_Float16 hl, _Float16 hh, int steps, int q, int i, bool &finite)
{
#pragma clang fp contract(off)
    const _Float16 e0 = line_space(hl, hh, S + 1, q), e1 = line_space(hl, hh, S + 1, q + 1);
    const _Float16 margin = fma_half(fabsf(static_cast<float>(e0)), 0.8f, 0.f);
    const _Float16 a0 = e0 - margin, a1 = e1 + margin;
    finite = finite && fabsf(static_cast<float>(a0)) < INFINITY && fabsf(static_cast<float>(a1)) < INFINITY;
    return line_space(a0, a1, steps, i);
}

struct SearchSpace {
    _Float16 scales[kEncMaxScales], axes[kEncMaxAxes];
    uint16_t group[kEncMaxG];
    float red[2][kEncThreads / 64];
    int scales_n, extended, covered;
};

// The bounds of the candidates of group m: its scales and axes into LDS, by the whole workgroup.
template <int S>
__device__ __forceinline__ void make_search_space(const sbvr_hip_encoder_run &a, const EncoderState &st, SearchSpace &sp)
{
#pragma clang fp contract(off)
    const int tid = threadIdx.x, m = st.miss;
    const uint16_t *mine = static_cast<const uint16_t *>(a.data) + static_cast<size_t>(m) * a.G;
    const float q95 = a.q95[m], mean = a.mean[m];                      // (asked for with the values, not behind the barrier)
    float lo = INFINITY, hi = -INFINITY;
    for (int i = tid; i < a.G; i += kEncThreads) {
        const uint16_t v = mine[i];
        sp.group[i] = v;
        lo = fminf(lo, h2f(v));
        hi = fmaxf(hi, h2f(v));
    }
    for (int d = 32; d >= 1; d >>= 1) {
        lo = fminf(lo, __shfl_xor(lo, d, 64));
        hi = fmaxf(hi, __shfl_xor(hi, d, 64));
    }
    if ((tid & 63) == 0) {
        sp.red[0][tid >> 6] = lo;
        sp.red[1][tid >> 6] = hi;
    }
    __syncthreads();
    for (int w = 0; w < kEncThreads / 64; ++w) {
        lo = fminf(lo, sp.red[0][w]);
        hi = fmaxf(hi, sp.red[1][w]);
    }
    const _Float16 hl = static_cast<_Float16>(lo), hh = static_cast<_Float16>(hi);
    const Scales scales = search_scales(a, st, q95, hl, hh);
    const int steps = a.axis_values[scales.wide];
    bool covered = fabsf(mean) * 2.f / S < 0.28f && scales.step != 0.f && scales.count > 0. && scales.count <= kEncMaxScales &&
                   st.lines < a.table_lines && fabsf(scales.from) < INFINITY && fabsf(lo) < INFINITY && fabsf(hi) < INFINITY;
    const int n = covered ? static_cast<int>(scales.count) : 0;
    for (int i = tid; i < n; i += kEncThreads)
        sp.scales[i] = fma_half(scales.step, static_cast<float>(i), scales.from);
    bool finite = true;
    for (int i = tid; i < S * steps; i += kEncThreads)
        sp.axes[i] = axis_value<S>(hl, hh, steps, i / steps, i % steps, finite);
    covered = __syncthreads_and(covered && finite);
    if (tid == 0) {
        sp.scales_n = n;
        sp.extended = scales.wide;
        sp.covered = covered;
    }
    __syncthreads();
}

// Quotient and remainder of numbers below 2^24 by a divisor that many share: a product, corrected.
struct Divider {
    uint32_t by;
    float reciprocal;
    __device__ __forceinline__ explicit Divider(int d) : by(static_cast<uint32_t>(d)), reciprocal(1.f / static_cast<float>(d)) {}
    __device__ __forceinline__ int operator()(int &x) const        // returns the quotient, leaves the remainder
    {
        int q = static_cast<int>(static_cast<float>(x) * reciprocal), rest = x - static_cast<int>(__umul24(static_cast<uint32_t>(q), by));
        q += rest < 0 ? -1 : (rest >= static_cast<int>(by) ? 1 : 0);
        rest += rest < 0 ? static_cast<int>(by) : (rest >= static_cast<int>(by) ? -static_cast<int>(by) : 0);
        x = rest;
        return q;
    }
};

struct Dividers {
    Divider bases, scales, steps;
};

// Candidate `at` (see sbvr_encoder_candidates_kernel for the order).  kSmall: there are fewer than 2^24.
template <int S, bool kSmall>
__device__ __forceinline__ void form_candidate(const sbvr_hip_encoder_run &a, const SearchSpace &sp, const Dividers &by, int family, int at,
                                               _Float16 (&c)[S])
{
#pragma clang fp contract(off)
    auto divide = [](int &x, const Divider &d) __attribute__((always_inline)) -> int {
        if constexpr (kSmall)
            return d(x);
        const int q = x / static_cast<int>(d.by);
        x -= q * static_cast<int>(d.by);
        return q;
    };
    const int wide = sp.extended, steps = static_cast<int>(by.steps.by);
    if (at < family) {
        const _Float16 *base = static_cast<const _Float16 *>(a.base[wide]), *offsets = static_cast<const _Float16 *>(a.offsets[wide]);
        int ir = at, is = divide(ir, by.bases), ib = divide(is, by.scales);
        const _Float16 sv = sp.scales[is], bv = offsets[ib];
#pragma unroll
        for (int q = 0; q < S; ++q) {
            const _Float16 scaled = sv * base[ir * S + q];
            c[q] = bv + scaled;
        }
    } else {
        int rest = at - family;
#pragma unroll
        for (int q = S - 1; q >= 0; --q) {
            int i = rest;
            rest = divide(i, by.steps);
            c[q] = sp.axes[q * steps + i];
        }
    }
}

// The 2^S subset sums of a line as packed pairs, entry i the sum of the coefficients of i's bits (fp32, rounded once).
template <int S>
__device__ __forceinline__ void subset_sums(const _Float16 (&c)[S], v2h (&p)[1 << (S - 1)])
{
#pragma clang fp contract(off)
    float sums[1 << S];
    sums[0] = 0.f;
#pragma unroll
    for (int q = 0; q < S; ++q)
#pragma unroll
        for (int i = 0; i < (1 << q); ++i)
            sums[(1 << q) + i] = sums[i] + static_cast<float>(c[q]);
#pragma unroll
    for (int j = 0; j < (1 << (S - 1)); ++j)
        p[j] = v2h{static_cast<_Float16>(sums[2 * j]), static_cast<_Float16>(sums[2 * j + 1])};
}

// The least squared distance of a value to the points: fp16 difference, fp16 square, and a packed minimum of three (which
// gives NaN for NaN: the values are finite here, and the points' sums at most infinite).  With v_pk_min_f16 four operations more of 25.
template <int S>
__device__ __forceinline__ float least_square(uint16_t raw, const v2h (&p)[1 << (S - 1)])
{
#pragma clang fp contract(off)
    const _Float16 d = __builtin_bit_cast(_Float16, raw);
    const v2h dd = {d, d};
    auto square = [&](int j) __attribute__((always_inline)) -> v2h {
        const v2h diff = dd - p[j];
        return diff * diff;
    };
    v2h best = __builtin_elementwise_min(square(0), square(1));
#pragma unroll
    for (int j = 2; j < (1 << (S - 1)); j += 2) {
        const v2h one = square(j), two = square(j + 1);
        asm("v_pk_minimum3_f16 %0, %0, %1, %2" : "+v"(best) : "v"(one), "v"(two));
    }
    return static_cast<float>(best[0] < best[1] ? best[0] : best[1]);
}

// Selectors of a group's values against a line: the first nearest of its points, most significant plane first.
template <int S>
__device__ __forceinline__ void write_selectors(const uint16_t *group, int G, const _Float16 (&c)[S], int *out)
{
#pragma clang fp contract(off)
    _Float16 p[1 << S];
#pragma unroll
    for (int i = 0; i < (1 << S); ++i) {
        float sum = 0.f;
#pragma unroll
        for (int j = 0; j < S; ++j)
            sum += (i >> (S - 1 - j)) & 1 ? static_cast<float>(c[j]) : 0.f;
        p[i] = static_cast<_Float16>(sum);
    }
    for (int g = threadIdx.x; g < G; g += kEncThreads) {
        const _Float16 d = __builtin_bit_cast(_Float16, group[g]);
        int sel = 0;
        _Float16 least{};
#pragma unroll
        for (int i = 0; i < (1 << S); ++i) {
            const _Float16 diff = d - p[i], sq = diff * diff;
            if (i == 0 || sq < least) {
                least = sq;
                sel = i;
            }
        }
        out[g] = sel;
    }
}

template <int S, bool kSmall>
__device__ __forceinline__ void search_candidates(const sbvr_hip_encoder_run &a, const SearchSpace &sp, float known,
                                                  unsigned long long *found, unsigned long long *least)
{
    const int tid = threadIdx.x, wide = sp.extended;
    const int family = a.bases[wide] * a.n_offsets[wide] * sp.scales_n;
    const Dividers by{Divider(a.bases[wide]), Divider(sp.scales_n), Divider(a.axis_values[wide])};
    int n = family, grid = 1;
#pragma unroll
    for (int q = 0; q < S; ++q)
        grid *= a.axis_values[wide];
    n += grid;
    // (more lines than the launch has threads, which the host's bound on the scales rules out, would go round again)
    for (int first = blockIdx.x * kEncThreads; first < n; first += gridDim.x * kEncThreads) {
        const int line = first + tid, at = min(line, n - 1);
        _Float16 c[S];
        form_candidate<S, kSmall>(a, sp, by, family, at, c);
        v2h p[1 << (S - 1)];
        subset_sums<S>(c, p);
        // no candidate above the best error known counts; the margin covers the division by G
        const unsigned long long now = __hip_atomic_load(found, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const float bound = now == ~0ull ? known : fminf(known, __uint_as_float(static_cast<uint32_t>(now >> 32)));
        const float limit = bound * static_cast<float>(a.G) * 1.000001f;
        float sum = 0.f;
        int g = 0;
        for (; g < a.G; g += 4) {                                  // (G is a multiple of 4)
            const uint2 four = *reinterpret_cast<const uint2 *>(sp.group + g);
            sum += least_square<S>(static_cast<uint16_t>(four.x), p);
            sum += least_square<S>(static_cast<uint16_t>(four.x >> 16), p);
            sum += least_square<S>(static_cast<uint16_t>(four.y), p);
            sum += least_square<S>(static_cast<uint16_t>(four.y >> 16), p);
            if (((g & 4) || g < 16) && __all(sum > limit))
                break;
        }
        const float mse = sum / static_cast<float>(a.G);
        unsigned long long key = g >= a.G && line < n && mse < known ? (static_cast<unsigned long long>(__float_as_uint(mse)) << 32) | static_cast<uint32_t>(line)
                                                                      : ~0ull;
        for (int d = 32; d >= 1; d >>= 1) {
            const unsigned long long other = __shfl_xor(key, d, 64);
            key = other < key ? other : key;
        }
        __syncthreads();
        if ((tid & 63) == 0)
            least[tid >> 6] = key;
        __syncthreads();
        if (tid == 0) {
            for (int w = 1; w < kEncThreads / 64; ++w)
                key = least[w] < key ? least[w] : key;
            if (key != ~0ull)
                atomicMin(found, key);
        }
    }
}

template <int S>
__global__ void __launch_bounds__(kEncThreads)
sbvr_encoder_search_kernel(const sbvr_hip_encoder_run a, int slot)
{
    __shared__ __align__(16) SearchSpace sp;
    __shared__ unsigned long long least[kEncThreads / 64];
    EncoderState *const states = static_cast<EncoderState *>(a.state);
    const EncoderState st = states[slot];
    const int have_met = a.groups - st.unmet;
    const bool idle = st.status != 0 || st.miss >= have_met, extends = st.status == 0 && idle && have_met < a.groups;
    const int tid = threadIdx.x;
    const float known = idle || st.lines < a.warmup ? INFINITY : a.best[st.miss];
    if (!idle)
        make_search_space<S>(a, st, sp);
    if (blockIdx.x == 0 && tid == 0) {
        // the other slot: what the settling launch finds there before it takes minima
        const bool stays = idle ? !extends : !sp.covered;
        states[slot ^ 1].miss = stays ? st.miss : kEncNone;
        states[slot ^ 1].found = ~0ull;
    }
    if (idle || !sp.covered)
        return;
    const int wide = sp.extended;
    long lines = static_cast<long>(a.bases[wide]) * a.n_offsets[wide] * sp.scales_n, grid = 1;
#pragma unroll
    for (int q = 0; q < S; ++q)
        grid *= a.axis_values[wide];
    if (lines + grid < (1 << 24))
        search_candidates<S, true>(a, sp, known, &states[slot].found, least);
    else
        search_candidates<S, false>(a, sp, known, &states[slot].found, least);
}

// The cut-off over the last errors, added up in the host's order; `last`: one that is not in the history yet.
__device__ __forceinline__ double cut_off(const sbvr_hip_encoder_run &a, int history, bool with_last, double last, double *part)
{
#pragma clang fp contract(off)
    const int len = min(history, a.window), from = history - len;
    double sum = 0.;
    for (int i0 = 0; i0 < len; i0 += kEncThreads) {
        __syncthreads();
        const int i = i0 + static_cast<int>(threadIdx.x);
        if (i < len)
            part[threadIdx.x] = with_last && from + i == history - 1 ? last : a.history[from + i];
        __syncthreads();
        for (int k = 0; k < min(kEncThreads, len - i0); ++k)
            sum += part[k];
    }
    const double cutoff = sum / len * 0.99;
    return cutoff < a.acceptable ? a.acceptable : cutoff;
}

// The winner of the search of group m = st.miss, its coefficients by magnitude, equal ones in their order.  Every wave works
// it out for itself.
template <int S>
__device__ __forceinline__ void winner(const sbvr_hip_encoder_run &a, const EncoderState &st, _Float16 (&c)[S])
{
#pragma clang fp contract(off)
    const uint16_t *mine = static_cast<const uint16_t *>(a.data) + static_cast<size_t>(st.miss) * a.G;
    const float q95 = a.q95[st.miss];
    float lo = INFINITY, hi = -INFINITY;
    for (int i = threadIdx.x & 63; i < a.G; i += 64) {
        lo = fminf(lo, h2f(mine[i]));
        hi = fmaxf(hi, h2f(mine[i]));
    }
    for (int d = 32; d >= 1; d >>= 1) {
        lo = fminf(lo, __shfl_xor(lo, d, 64));
        hi = fmaxf(hi, __shfl_xor(hi, d, 64));
    }
    const _Float16 hl = static_cast<_Float16>(lo), hh = static_cast<_Float16>(hi);
    const Scales scales = search_scales(a, st, q95, hl, hh);
    const int wide = scales.wide, bases = a.bases[wide], steps = a.axis_values[wide], n = static_cast<int>(scales.count);
    const int family = bases * a.n_offsets[wide] * n, at = static_cast<int>(st.found & 0xffffffffu);
    _Float16 raw[S];
    if (at < family) {
        const _Float16 *base = static_cast<const _Float16 *>(a.base[wide]) + static_cast<size_t>(at % bases) * S;
        const _Float16 sv = fma_half(scales.step, static_cast<float>(at / bases % n), scales.from);
        const _Float16 bv = static_cast<const _Float16 *>(a.offsets[wide])[at / bases / n];
#pragma unroll
        for (int q = 0; q < S; ++q) {
            const _Float16 scaled = sv * base[q];
            raw[q] = bv + scaled;
        }
    } else {
        int rest = at - family;
        bool finite = true;
#pragma unroll
        for (int q = S - 1; q >= 0; --q) {
            raw[q] = axis_value<S>(hl, hh, steps, q, rest % steps, finite);
            rest /= steps;
        }
    }
#pragma unroll
    for (int q = 0; q < S; ++q) {
        int rank = 0;
#pragma unroll
        for (int o = 0; o < S; ++o) {
            const float vo = fabsf(static_cast<float>(raw[o])), vq = fabsf(static_cast<float>(raw[q]));
            rank += vo < vq || (vo == vq && o < q);
        }
#pragma unroll
        for (int o = 0; o < S; ++o)
            c[o] = rank == o ? raw[q] : c[o];
    }
}

// The next groups meet the whole table: a workgroup a group, a thread every 256th line; the least error and the first line
// that has it.
template <int S>
__device__ __forceinline__ void meet_table(const sbvr_hip_encoder_run &a, const EncoderState &st, int have_met, EncoderState *other,
                                           uint16_t *group, unsigned long long *least, double *part)
{
    const int tid = threadIdx.x, end = min(a.groups, have_met + kEncWindow);
    const bool looks = st.lines >= a.warmup;
    const double cutoff = looks ? cut_off(a, st.history, false, 0., part) : 0.;
    if (blockIdx.x == 0 && tid == 0) {
        other->lines = st.lines;
        other->misses = st.misses;
        other->history = st.history;
        other->status = 0;
        other->unmet = a.groups - end;
        atomicMin(&other->miss, looks ? end : have_met);
    }
    for (int g = have_met + static_cast<int>(blockIdx.x); g < end; g += static_cast<int>(gridDim.x)) {
        __syncthreads();
        for (int i = tid; i < a.G; i += kEncThreads)
            group[i] = static_cast<const uint16_t *>(a.data)[static_cast<size_t>(g) * a.G + i];
        __syncthreads();
        unsigned long long key = (static_cast<unsigned long long>(__float_as_uint(INFINITY)) << 32) | 0xffffffffu;
        for (int l = tid; l < st.lines; l += kEncThreads) {
            _Float16 c[S];
#pragma unroll
            for (int q = 0; q < S; ++q)
                c[q] = static_cast<const _Float16 *>(a.table)[static_cast<size_t>(l) * S + q];
            v2h p[1 << (S - 1)];
            subset_sums<S>(c, p);
            float sum = 0.f;
            for (int i = 0; i < a.G; i += 4) {
                const uint2 four = *reinterpret_cast<const uint2 *>(group + i);
                sum += least_square<S>(static_cast<uint16_t>(four.x), p);
                sum += least_square<S>(static_cast<uint16_t>(four.x >> 16), p);
                sum += least_square<S>(static_cast<uint16_t>(four.y), p);
                sum += least_square<S>(static_cast<uint16_t>(four.y >> 16), p);
            }
            const float mse = sum / static_cast<float>(a.G);
            if (mse < __uint_as_float(static_cast<uint32_t>(key >> 32)))
                key = (static_cast<unsigned long long>(__float_as_uint(mse)) << 32) | static_cast<uint32_t>(l);
        }
        for (int d = 32; d >= 1; d >>= 1) {
            const unsigned long long o = __shfl_xor(key, d, 64);
            key = o < key ? o : key;
        }
        if ((tid & 63) == 0)
            least[tid >> 6] = key;
        __syncthreads();
        if (tid == 0) {
            for (int w = 1; w < kEncThreads / 64; ++w)
                key = least[w] < key ? least[w] : key;
            const float best = __uint_as_float(static_cast<uint32_t>(key >> 32));
            a.best[g] = best;
            a.line[g] = static_cast<int>(static_cast<uint32_t>(key));      // (-1 without a line)
            if (looks && !(static_cast<double>(best) < cutoff))
                atomicMin(&other->miss, g);
        }
    }
}

template <int S>
__global__ void __launch_bounds__(kEncThreads)
sbvr_encoder_settle_kernel(const sbvr_hip_encoder_run a, int slot)
{
#pragma clang fp contract(off)
    __shared__ __align__(16) union {
        uint16_t group[kEncMaxG];
        float squares[kEncMaxG + 64];
    } sh;
    __shared__ double part[kEncThreads];
    __shared__ unsigned long long least[kEncThreads / 64];
    __shared__ int twin, first_miss;
    EncoderState *const states = static_cast<EncoderState *>(a.state), *const other = &states[slot ^ 1];
    const EncoderState st = states[slot];
    const int have_met = a.groups - st.unmet;
    const int tid = threadIdx.x, m = st.miss;
    _Float16 *const table = static_cast<_Float16 *>(a.table);
    if (st.status == 0 && m >= have_met && have_met < a.groups) {
        meet_table<S>(a, st, have_met, other, sh.group, least, part);
        return;
    }
    EncoderState next = st;                                            // (miss and found: written by the search and by minima)
    const bool found = st.found != ~0ull;
    // (nothing left, a group for the host, or one that neither the table nor any candidate has an error for: the state stays)
    const bool uncovered = m < a.groups && other->miss == m;            // (what this launch takes minima of is behind m; or m, unserved)
    const bool stays = st.status != 0 || m >= a.groups || uncovered, unserved = !stays && !found && a.line[m] < 0;
    if (stays || unserved) {
        if (blockIdx.x == 0 && tid == 0) {
            other->lines = st.lines;
            other->misses = st.misses;
            other->history = st.history;
            other->unmet = st.unmet;
            other->status = unserved || uncovered ? 1 : st.status;
            if (unserved)
                atomicMin(&other->miss, m);
        }
        return;
    }
    const int per = max(1, kEncSettleValues / a.G), stride = a.G + 4;
    if (blockIdx.x > 0 && m + 1 + static_cast<int>(blockIdx.x) * per >= have_met)      // (nothing to show the line to; warming up or not)
        return;
    _Float16 c[S];
    if (found) {
        winner<S>(a, st, c);
    } else {
        const _Float16 *have = table + static_cast<size_t>(a.line[m]) * S;
#pragma unroll
        for (int q = 0; q < S; ++q)
            c[q] = have[q];
    }
    if (tid == 0)
        twin = kEncNone;
    __syncthreads();
    // a line of the table that is the same but for 1e-4 takes its place
    if (found) {
        float size = 0.f;
#pragma unroll
        for (int q = 0; q < S; ++q)
            size += fabsf(static_cast<float>(c[q]));
        const _Float16 bound = fma_half(static_cast<float>(static_cast<_Float16>(size)), 0.0001f, 0.f);
        for (int l = tid; l < st.lines; l += kEncThreads) {
            float off = 0.f;
#pragma unroll
            for (int q = 0; q < S; ++q)
                off += fabsf(static_cast<float>(static_cast<_Float16>(table[static_cast<size_t>(l) * S + q] - c[q])));
            if (static_cast<_Float16>(off) < bound) {
                atomicMin(&twin, l);
                break;
            }
        }
    }
    __syncthreads();
    const bool joins = found && twin == kEncNone;
    const int chosen = !found ? a.line[m] : (joins ? st.lines : twin);
    const double error = static_cast<double>(__uint_as_float(static_cast<uint32_t>(st.found >> 32)));
    next.lines = st.lines + joins;
    next.misses = st.misses + 1;
    next.history = st.history + found;
    const double cutoff = cut_off(a, next.history, found, error, part);
    if (blockIdx.x == 0) {
        write_selectors<S>(static_cast<const uint16_t *>(a.data) + static_cast<size_t>(m) * a.G, a.G, c, a.sel + static_cast<size_t>(m) * a.G);
        if (tid == 0) {
            a.line_of[m] = chosen;
            a.settled[m] = 1;
            if (joins)
#pragma unroll
                for (int q = 0; q < S; ++q)
                    table[static_cast<size_t>(st.lines) * S + q] = c[q];
            if (found)
                a.history[st.history] = error;
            other->lines = next.lines;
            other->misses = next.misses;
            other->history = next.history;
            other->unmet = st.unmet;
            other->status = 0;
            // (groups are searched one after the other until the table has its first lines)
            atomicMin(&other->miss, next.lines < a.warmup ? m + 1 : have_met);
        }
    }
    const bool looks = next.lines >= a.warmup;
    if (!joins && !looks)
        return;
    v2h p[1 << (S - 1)];
    subset_sums<S>(c, p);
    for (int g0 = m + 1 + static_cast<int>(blockIdx.x) * per; g0 < have_met; g0 += static_cast<int>(gridDim.x) * per) {
        const int many = min(per, have_met - g0);
        __syncthreads();
        if (tid == 0)
            first_miss = kEncNone;
        if (joins)
            for (int i = tid; i < many * a.G; i += kEncThreads)
                sh.squares[i / a.G * stride + i % a.G] = least_square<S>(static_cast<const uint16_t *>(a.data)[static_cast<size_t>(g0) * a.G + i], p);
        __syncthreads();
        if (tid < many) {
            const int g = g0 + tid;
            float best = a.best[g];
            if (joins) {
                float sum = 0.f;
#pragma unroll 8
                for (int i = 0; i < a.G; i += 4) {                     // (element order)
                    const v4f four = *reinterpret_cast<const v4f *>(sh.squares + tid * stride + i);
                    sum += four.x;
                    sum += four.y;
                    sum += four.z;
                    sum += four.w;
                }
                const float mse = sum / static_cast<float>(a.G);
                if (mse < best) {
                    best = mse;
                    a.best[g] = mse;
                    a.line[g] = chosen;
                }
            }
            if (looks && !(static_cast<double>(best) < cutoff))
                atomicMin(&first_miss, g);
        }
        __syncthreads();
        if (tid == 0 && first_miss != kEncNone)
            atomicMin(&other->miss, first_miss);
    }
}

// Selectors of the groups that a table line serves: a workgroup a group.
template <int S>
__global__ void __launch_bounds__(kEncThreads)
sbvr_encoder_selectors_kernel(const sbvr_hip_encoder_run a, int first, int groups)
{
    __shared__ __align__(16) uint16_t group[kEncMaxG];
    for (int g = first + static_cast<int>(blockIdx.x); g < first + groups; g += static_cast<int>(gridDim.x)) {
        if (a.settled[g])                                          // (the same for the whole workgroup)
            continue;
        __syncthreads();
        for (int i = threadIdx.x; i < a.G; i += kEncThreads)
            group[i] = static_cast<const uint16_t *>(a.data)[static_cast<size_t>(g) * a.G + i];
        __syncthreads();
        _Float16 c[S];
#pragma unroll
        for (int q = 0; q < S; ++q)
            c[q] = static_cast<const _Float16 *>(a.table)[static_cast<size_t>(max(a.line[g], 0)) * S + q];
        write_selectors<S>(group, a.G, c, a.sel + static_cast<size_t>(g) * a.G);
        if (threadIdx.x == 0)
            a.line_of[g] = a.line[g];
    }
}

template <int S>
void launch_rounds(const sbvr_hip_encoder_run &a, unsigned search_grid, int slot, int rounds, hipStream_t st)
{
    // (a workgroup for two groups that meet the table; showing them one line takes a quarter of these: with 1024 at work on that
    // it took 13 to 16 us, 8 so)
    const unsigned settle_grid = static_cast<unsigned>(max(1, (min(a.groups, kEncWindow) + 1) / 2));
    for (int r = 0; r < rounds; ++r) {
        hipLaunchKernelGGL(sbvr_encoder_search_kernel<S>, dim3(search_grid), dim3(kEncThreads), 0, st, a, (slot + r) & 1);
        hipLaunchKernelGGL(sbvr_encoder_settle_kernel<S>, dim3(settle_grid), dim3(kEncThreads), 0, st, a, (slot + r) & 1);
    }
}

template <int S>
void launch_selectors(const sbvr_hip_encoder_run &a, int first, int groups, hipStream_t st)
{
    hipLaunchKernelGGL(sbvr_encoder_selectors_kernel<S>, dim3(static_cast<unsigned>(min(groups, 8192))), dim3(kEncThreads), 0, st, a, first, groups);
}

bool run_ok(const sbvr_hip_encoder_run *a)
{
    return a && a->data && a->q95 && a->mean && a->table && a->best && a->line && a->line_of && a->sel && a->settled && a->state && a->history &&
           a->base[0] && a->base[1] && a->offsets[0] && a->offsets[1] && a->groups > 0 && a->G > 0 && a->bases[0] > 0 && a->bases[1] > 0 &&
           a->n_offsets[0] > 0 && a->n_offsets[1] > 0 && a->axis_values[0] > 1 && a->axis_values[1] > 1 && a->window > 0 && a->warmup > 0 &&
           a->table_lines > 0;
}

// The lines of a search of the wider or the plainer kind, at most; 0 where the kernels have no room for it.
long run_lines(const sbvr_hip_encoder_run &a, int wide, int S)
{
    if (static_cast<long>(S) * a.axis_values[wide] > kEncMaxAxes)
        return 0;
    double grid = 1.;
    for (int q = 0; q < S; ++q)
        grid *= a.axis_values[wide];
    const double n = static_cast<double>(a.bases[wide]) * a.n_offsets[wide] * kEncMaxScales + grid;
    return n < (1 << 28) ? static_cast<long>(n) : 0;
}

// Activations to bit planes on the fly: lane = one element x[m, k]; its selector is the first of the P
// subset sums of its group's line that is nearest to it (fp16 difference and square, as the encoder chooses
// selectors: sbvr/core.py:492-494), and the 64 lanes' selector bits become two words per plane by ballot
// (a selector counts the subset sums most significant coefficient first: plane j is its bit S - 1 - j,
// core.py:345-351 and :842-876).
// A workgroup takes 64 elements of K (two words) of kOnlineRows rows, one row a wave at a time, and keeps the subset
// sums of the (at most two) groups they lie in in LDS, where the waves read them four pairs at a time: built from
// the group's coefficients (kLines: each the fp32 sum in the order of the planes, rounded to fp16 once), or copied
// from a table of them.  The search is the vector ALU's: per two points a packed difference and square, then each
// square's bits above its point's number as one key (squares are not negative: their bits order as they do) and a
// three-way minimum, 2.5 operations a point.  (16 rows x 4096, 256 points: the lane that fetched every point from
// memory for itself took 20.5 us.)
constexpr int kOnlineWaves = 4, kOnlineRows = 4;
constexpr float kOnlineCoarse = 1.5f * 134217728.f;       // 1.5 x 2^27, whose neighbours are 2^4 away

// kImage: also the encoded values as the A operands of sbvr_online_product_kernel (OnlineArgs), and a scale per group: the
// power of two that puts the sum of the line's magnitudes below 2^15.
template <bool kLines, bool kImage>
__global__ void __launch_bounds__(64 * kOnlineWaves)
sbvr_online_encode_kernel(const uint16_t *__restrict__ x, const uint16_t *__restrict__ table, uint32_t *__restrict__ bvr,
                          uint8_t *__restrict__ idx, int idx16, int M, int K, int G, int S, uint32_t *__restrict__ image,
                          float *__restrict__ scales)
{
    __shared__ __align__(16) uint16_t pts[2][256];
    __shared__ float sums[kImage ? 2 : 1][kImage ? 256 : 1], ups[2];      // the points before their rounding, the powers of two
    __shared__ float coeffs[2][8];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int P = 1 << S, padded = max(P, 8);
    const int k0 = blockIdx.x * 64;
    const int words = K / 32;
    const int groups = K / G, g0 = k0 / G, g1 = min((k0 + 32) / G, groups - 1);     // (G is a multiple of 32)
    const int k = min(k0 + lane, K - 1);
    static_assert(kOnlineRows == kOnlineWaves, "a row a wave");
    const int m = blockIdx.y * kOnlineRows + wave;
    // (everything asked for at once: the activation, and a coefficient a thread; fetched in the loop over the planes below, the
    // coefficients alone took 2 us)
    const _Float16 d = __builtin_bit_cast(_Float16, x[static_cast<size_t>(min(m, M - 1)) * K + k]);
    if constexpr (kLines) {
        if (threadIdx.x < 16 && (threadIdx.x & 7) < S)
            coeffs[threadIdx.x >> 3][threadIdx.x & 7] = h2f(table[static_cast<size_t>(threadIdx.x >> 3 ? g1 : g0) * S + (threadIdx.x & 7)]);
        __syncthreads();
    }
    for (int i = threadIdx.x; i < 2 * padded; i += 64 * kOnlineWaves) {
        const int which = i >= padded, p = min(which ? i - padded : i, P - 1);       // (the last point again behind the end)
        const int g = which ? g1 : g0;
        uint16_t v;
        if constexpr (kLines) {
            float sum = 0.f;
            for (int j = 0; j < S; ++j) {
                const float c = coeffs[which][j];
                sum += (p >> (S - 1 - j)) & 1 ? c : 0.f * c;       // (NaN where c is not finite, as a product would have it)
            }
            v = f2h(sum);
            if constexpr (kImage) {
                if ((which ? i - padded : i) < P)
                    sums[which][p] = sum;
                if (p == 0) {
                    float size = 0.f;
                    for (int j = 0; j < S; ++j)
                        size += fabsf(coeffs[which][j]);
                    // At least 2^-24 and below 2^19, or zero.  Or not finite: then the group's first point is NaN, every value
                    // selects it, and no bit at all times that coefficient is NaN in every output.
                    const int exponent = static_cast<int>(__float_as_uint(size) >> 23);
                    const int up = exponent == 255 || exponent == 0 ? 0 : 141 - exponent;
                    ups[which] = __uint_as_float(static_cast<uint32_t>(127 + up) << 23);
                    if (blockIdx.y == 0)
                        scales[g] = exponent == 255 ? NAN : __uint_as_float(static_cast<uint32_t>(127 + 14 - up) << 23);
                }
            }
        } else {
            v = table[static_cast<size_t>(g) * P + p];
        }
        pts[which][which ? i - padded : i] = v;
    }
    __syncthreads();
    const uint4 *const mine = reinterpret_cast<const uint4 *>(pts[lane >> 5 & (g1 != g0)]);
    if (m < M) {                                                                      // wave-uniform
        const v2h dd = {d, d};
        uint32_t best = 0xffffffffu;
#pragma unroll 4
        for (int c = 0; c < padded / 8; ++c) {
            const uint4 q = mine[c];
            const uint32_t w[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const v2h diff = dd - __builtin_bit_cast(v2h, w[i]);
                const uint32_t sq = __builtin_bit_cast(uint32_t, diff * diff);
                const uint32_t p = static_cast<uint32_t>(8 * c + 2 * i);
                best = min(min(best, (sq << 16) | p), (sq & 0xffff0000u) | (p + 1));
            }
        }
        // (a distance that is no number is never the nearest, but the first of them stays: the search starts with it)
        const _Float16 d0 = d - __builtin_bit_cast(v2h, mine[0].x)[0], first = d0 * d0;
        const uint32_t sel = first != first ? 0u : best & 0xffffu;
        uint32_t out = 0;
        for (int j = 0; j < S; ++j) {                                                 // plane 0: the selector's top bit
            const unsigned long long bits = __builtin_amdgcn_ballot_w64(((sel >> (S - 1 - j)) & 1) != 0);
            out = (lane & 31) == j ? static_cast<uint32_t>(lane < 32 ? bits : bits >> 32) : out;
        }
        if constexpr (kImage) {                                                       // (K is a multiple of 128)
            const int at = k0 + lane, i = at & 15, which = lane >> 5 & (g1 != g0);
            const float v = sums[which][sel] * ups[which], by = __uint_as_float(static_cast<uint32_t>(128 - (1 << online_bit(i))) << 23);
            const float tall = v + kOnlineCoarse - kOnlineCoarse;                     // (a multiple of 2^4)
            const _Float16 head = static_cast<_Float16>(tall * by), rest = static_cast<_Float16>((v - tall) * by);
            const uint32_t both = static_cast<uint32_t>(__builtin_bit_cast(uint16_t, head)) | static_cast<uint32_t>(__builtin_bit_cast(uint16_t, rest)) << 16;
            const uint32_t other = static_cast<uint32_t>(__shfl_xor(static_cast<int>(both), 16, 64));
            // lanes 0 to 15 of 32 store the pair's heads, lanes 16 to 31 the rests
            const int part = (lane >> 4) & 1;
            const uint32_t pair = part ? __builtin_amdgcn_perm(both, other, 0x07060302u) : __builtin_amdgcn_perm(other, both, 0x05040100u);
            const size_t tile = static_cast<size_t>(at >> 7) * ((M + 15) / 16) + (m >> 4);
            image[(((tile * 4 + (i >> 2)) * 2 + part) * 64 + ((at >> 5) & 3) * 16 + (m & 15)) * 4 + (i & 3)] = pair;
        }
        const int kw = blockIdx.x * 2 + (lane >> 5);
        if ((lane & 31) < S && kw < words)
            bvr[(static_cast<size_t>(kw) * M + m) * S + (lane & 31)] = out;
        // the left operand's line index of a group is the group's number
        if (idx && (lane & 31) == 31 && kw < words && kw * 32 % G == 0) {
            const int g = kw * 32 / G;
            if (idx16)
                reinterpret_cast<uint16_t *>(idx)[static_cast<size_t>(g) * M + m] = static_cast<uint16_t>(g);
            else
                idx[static_cast<size_t>(g) * M + m] = static_cast<uint8_t>(g);
        }
    }
}

// ------------------------------------------------------------------------------------ the dense weight again
//
// decode(): out[n, k] = the subset sum that the planes of (n, k) select from the line of n's group, the fp32 sum
// rounded to fp16 once (reference sbvr/core.py:926-949), then converted to the tensor's own type (OUT: fp16, bf16
// or fp32).  A wave takes 8 columns x 8 words of K: lane (n = lane % 8, word = lane / 8) loads its plane words (eight
// neighbouring columns of a word are one or two cache lines) and decodes 32 weights in registers, by table look-up
// for 2, 3 and 4 planes (S).  6 and 8 planes: two tables of fp32 sums a column in LDS, 8 or 16 entries each, where every such
// sum is exact whatever its order (the table lines of all the wave's columns say so); otherwise, and for any other number
// of planes (S = 0), plane by plane in fp32.  Eight words of a row are 512
// bytes of output; the 64-byte pieces of the lanes go through 4 KiB of LDS to lanes that follow each other along a
// row, so that a store instruction writes two runs of 512 bytes.  Bound by memory: 2 bytes out per weight against S / 8
// in.  An index beyond the table gives NaN (torch's indexing ends the process there).  4096 -> 14336, 4 planes: 29.6 us a call
// among others on weights that take turns = 5.0 TB/s, where a large copy reaches 5.2 (the torch expression over unpacked
// 64-bit selectors took 4.4 ms); 34.9 with the workgroups dealt out over the columns first, and 2 and 3 planes 22 and 23
// where that took 28 and 30.  (Stores that pass the caches by: 27.0, but a copy of the result then took 47 where it takes
// 33, so the caller would lose more than the call gains.)  6 and 8 planes: 32 and 40, plane by plane 67 and 82, bound by the
// vector ALU.
struct DecodeArgs {
    const uint32_t *bvr;
    const uint8_t *idx;
    const uint16_t *cache;
    void *out;
    int N, words, S, wpg, L, idx16;
    int k_out;                   // columns of the output: K without the padding
    int wide;                    // rows of the output are 16-byte aligned
};

constexpr int kDecWaves = 4;
enum { kOutF16 = 0, kOutBf16 = 1, kOutF32 = 2 };

__device__ __forceinline__ uint32_t bf16_pair(uint32_t two)
{
    auto one = [](uint16_t h) __attribute__((always_inline)) -> uint32_t {
        const uint32_t u = __float_as_uint(h2f(h));
        return (u & 0x7fffffffu) > 0x7f800000u ? 0x7fc0u : (u + 0x7fffu + ((u >> 16) & 1u)) >> 16;
    };
    return one(static_cast<uint16_t>(two & 0xffffu)) | (one(static_cast<uint16_t>(two >> 16)) << 16);
}

__device__ __forceinline__ bool not_finite(uint16_t h) { return (h & 0x7c00u) == 0x7c00u; }

template <int S, int OUT>
__global__ void __launch_bounds__(64 * kDecWaves)
sbvr_decode_weight_kernel(const DecodeArgs a)
{
    constexpr bool kSums = S > 4;                 // two tables of fp32 sums
    constexpr int H = kSums ? S / 2 : 4;          // planes of each
    __shared__ v4u tiles[kDecWaves][S == 8 ? 512 : 256];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    // Workgroups go to the 8 XCDs in turn: each takes a run of rows, along K first, so that what is written at one time is
    // whole rows, and a cache line of plane words or indices that two windows of columns share is read by one L2.
    unsigned lin = blockIdx.y * gridDim.x + blockIdx.x;
    const unsigned run = gridDim.x * gridDim.y / 8;
    if (lin < 8 * run)
        lin = lin % 8 * run + lin / 8;
    const int w0 = (lin % gridDim.y * kDecWaves + wave) * 8, n0 = lin / gridDim.y * 8;
    if (w0 >= a.words)                                        // wave-uniform; no barrier below
        return;
    v4u *const tile = tiles[wave];
    const int ln = lane & 7, lw = lane >> 3;
    const int n = min(n0 + ln, a.N - 1), word = min(w0 + lw, a.words - 1);
    const size_t at = (static_cast<size_t>(word / a.wpg) * a.N + n) << a.idx16;
    const int lo = a.idx[at], hi = a.idx[at + a.idx16];
    const int line_read = a.idx16 ? lo | (hi << 8) : lo, line = min(line_read, a.L - 1);
    uint32_t D[16];                                           // elements 2i, 2i + 1 of the word
    // any planes, in their order
    auto plane_by_plane = [&]() __attribute__((always_inline)) {
        float w[32];
#pragma unroll
        for (int i = 0; i < 32; ++i)
            w[i] = 0.f;
        const uint32_t *src = a.bvr + (static_cast<size_t>(word) * a.N + n) * a.S;
        const uint16_t *cs = a.cache + static_cast<size_t>(line) * a.S;
#pragma unroll 1
        for (int j = 0; j < a.S; ++j) {
            const int bits = static_cast<int>(src[j]);
            const uint32_t c = __float_as_uint(h2f(cs[j])), without = not_finite(cs[j]) ? 0x7fc00000u : 0u;   // (0 * c)
#pragma unroll
            for (int i = 0; i < 32; ++i) {
                const uint32_t set = static_cast<uint32_t>(__builtin_amdgcn_sbfe(bits, i, 1));
                w[i] += __uint_as_float((set & c) | (~set & without));
            }
        }
#pragma unroll
        for (int i = 0; i < 16; ++i)
            D[i] = static_cast<uint32_t>(f2h(w[2 * i])) | (static_cast<uint32_t>(f2h(w[2 * i + 1])) << 16);
    };
    if constexpr (kSums) {
        const Planes<S> pl = load_planes<S>(a.bvr + (static_cast<size_t>(word) * a.N + n) * S);
        uint32_t c[(S + 1) / 2];
        load_line_words<S>(a.cache + static_cast<size_t>(line) * S, c);
        // Coefficients are multiples of 2^(least - 25) below 2^(most - 14), by their exponents.  Where these differ by 10 at
        // most, a sum of eight is a number of 24 bits of that unit: exact, so in whatever order it is added up.
        float f[S];
        int most = 0, least = 31;
#pragma unroll
        for (int j = 0; j < S; ++j) {
            const uint16_t h = static_cast<uint16_t>(j & 1 ? c[j / 2] >> 16 : c[j / 2]);
            f[j] = h2f(h);
            const int e = max((h >> 10) & 31, 1);
            most = max(most, e);
            least = (h & 0x7fff) != 0 ? min(least, e) : least;
        }
        if (__all(most < 31 && most - least <= 10)) {
            // tables of the lane's own column: [low, high planes][sum][lane], no two lanes of a read in one bank
            float *const sums = reinterpret_cast<float *>(tile) + lane;
            uint32_t nibbles[2][4];           // nibble i of [.][p]: the planes' bits of element p + 4 i
#pragma unroll
            for (int half = 0; half < 2; ++half) {
                float s[1 << H];
                s[0] = 0.f;
#pragma unroll
                for (int b = 0; b < H; ++b)
#pragma unroll
                    for (int i = 0; i < 1 << b; ++i)
                        s[(1 << b) + i] = s[i] + f[half * H + b];
#pragma unroll
                for (int i = 0; i < 1 << H; ++i)
                    sums[((half << H) + i) * 64] = s[i];
                const uint32_t *const w = pl.w + half * H;
                const uint32_t w3 = H == 4 ? w[H - 1] : 0u;
                const uint32_t even = bit_select(0x55555555u, w[0], w[1] << 1), odd = bit_select(0x55555555u, w[0] >> 1, w[1]);
                const uint32_t even2 = bit_select(0x55555555u, w[2], w3 << 1), odd2 = bit_select(0x55555555u, w[2] >> 1, w3);
                nibbles[half][0] = bit_select(0x33333333u, even, even2 << 2);
                nibbles[half][1] = bit_select(0x33333333u, odd, odd2 << 2);
                nibbles[half][2] = bit_select(0x33333333u, even >> 2, even2);
                nibbles[half][3] = bit_select(0x33333333u, odd >> 2, odd2);
            }
            __builtin_amdgcn_wave_barrier();
            auto weight = [&](int p, int i) __attribute__((always_inline)) -> float {
                constexpr uint32_t kMask = (1u << H) - 1u;
                return sums[((nibbles[0][p] >> (4 * i)) & kMask) * 64] + sums[((nibbles[1][p] >> (4 * i)) & kMask) * 64 + (64 << H)];
            };
#pragma unroll
            for (int i = 0; i < 16; ++i)
                D[i] = static_cast<uint32_t>(f2h(weight(2 * (i & 1), i >> 1))) |
                       (static_cast<uint32_t>(f2h(weight(2 * (i & 1) + 1, i >> 1))) << 16);
            __builtin_amdgcn_wave_barrier();
        } else {
            plane_by_plane();
        }
    } else if constexpr (S != 0) {
        const Planes<S> pl = load_planes<S>(a.bvr + (static_cast<size_t>(word) * a.N + n) * S);
        uint32_t c[(S + 1) / 2];
        load_line_words<S>(a.cache + static_cast<size_t>(line) * S, c);
        LutTables<S> t;
        lut_build_tables<S>(c, t);
        Nibbles<S> Q;
        lut_nibble_words<S>(pl.w, Q);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            uint32_t e01, e23, o01, o23;                      // elements p, p + 8 and p + 16, p + 24
            lut_look_up<S>(t, Q, 2 * q, e01, e23);
            lut_look_up<S>(t, Q, 2 * q + 1, o01, o23);
            D[q] = __builtin_amdgcn_perm(o01, e01, 0x05040100u);
            D[4 + q] = __builtin_amdgcn_perm(o01, e01, 0x07060302u);
            D[8 + q] = __builtin_amdgcn_perm(o23, e23, 0x05040100u);
            D[12 + q] = __builtin_amdgcn_perm(o23, e23, 0x07060302u);
        }
        // an infinite or NaN coefficient counts in the elements that do not select it too, as 0 * inf = NaN
        uint32_t poison = 0;
#pragma unroll
        for (int j = 0; j < S; ++j)
            if (not_finite(static_cast<uint16_t>(j & 1 ? c[j / 2] >> 16 : c[j / 2])))
                poison |= ~pl.w[j];
        if (poison) {
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                D[i] = (poison >> (2 * i)) & 1u ? (D[i] & 0xffff0000u) | 0x7e00u : D[i];
                D[i] = (poison >> (2 * i + 1)) & 1u ? (D[i] & 0xffffu) | 0x7e000000u : D[i];
            }
        }
    } else {
        plane_by_plane();
    }
    if (line_read >= a.L)
#pragma unroll
        for (int i = 0; i < 16; ++i)
            D[i] = 0x7e007e00u;
    // 16-byte piece c of word w of row n lies at place (w ^ n) * 4 + c of the row's 32: the lanes that read a row meet
    // different banks; eight lanes that store piece c of one word of eight rows still share a quarter of them (24 clocks
    // more a store by SQ_LDS_BANK_CONFLICT, in the shadow of memory)
#pragma unroll
    for (int c = 0; c < 4; ++c)
        tile[ln * 32 + ((lw ^ ln) << 2) + c] = v4u{D[4 * c], D[4 * c + 1], D[4 * c + 2], D[4 * c + 3]};
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        const int row = 2 * s + (lane >> 5), q = lane & 31;
        v4u v = tile[row * 32 + (((q >> 2) ^ row) << 2) + (q & 3)];
        if constexpr (OUT == kOutBf16) {
#pragma unroll
            for (int i = 0; i < 4; ++i)
                v[i] = bf16_pair(v[i]);
        }
        const int k = w0 * 32 + 8 * q, nn = n0 + row;
        if (nn >= a.N || k >= a.k_out)
            continue;
        const size_t o = static_cast<size_t>(nn) * a.k_out + k;
        if (a.wide && k + 8 <= a.k_out) {
            if constexpr (OUT == kOutF32) {
                float *dst = static_cast<float *>(a.out) + o;
#pragma unroll
                for (int i = 0; i < 2; ++i)
                    *reinterpret_cast<v4f *>(dst + 4 * i) =
                        v4f{h2f(static_cast<uint16_t>(v[2 * i])), h2f(static_cast<uint16_t>(v[2 * i] >> 16)),
                            h2f(static_cast<uint16_t>(v[2 * i + 1])), h2f(static_cast<uint16_t>(v[2 * i + 1] >> 16))};
            } else {
                *reinterpret_cast<v4u *>(static_cast<uint16_t *>(a.out) + o) = v;
            }
        } else {
#pragma unroll
            for (int i = 0; i < 8; ++i)
                if (k + i < a.k_out) {
                    const uint16_t h = static_cast<uint16_t>(v[i / 2] >> (16 * (i & 1)));
                    if constexpr (OUT == kOutF32)
                        static_cast<float *>(a.out)[o + i] = h2f(h);
                    else
                        static_cast<uint16_t *>(a.out)[o + i] = h;
                }
        }
    }
}

template <int S>
void launch_decode(int out_type, dim3 grid, hipStream_t st, const DecodeArgs &a)
{
    const dim3 block(64 * kDecWaves);
    if (out_type == kOutF16)
        hipLaunchKernelGGL((sbvr_decode_weight_kernel<S, kOutF16>), grid, block, 0, st, a);
    else if (out_type == kOutBf16)
        hipLaunchKernelGGL((sbvr_decode_weight_kernel<S, kOutBf16>), grid, block, 0, st, a);
    else
        hipLaunchKernelGGL((sbvr_decode_weight_kernel<S, kOutF32>), grid, block, 0, st, a);
}

int device_cus()
{
    int device = 0, cus = 0;
    return hipGetDevice(&device) == hipSuccess && hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) == hipSuccess ? cus : 256;
}

}  // namespace

extern "C" {

int sbvr_hip_encoder_group_mse_f16(const void *data, const void *points, float *mse, int groups, int G, int n, int P,
                                   void *stream)
{
    if (!data || !points || !mse || groups <= 0 || G <= 0 || n <= 0)
        return -1;
    if (groups > 65535 || P < 2 || P > 256 || (P & (P - 1)) != 0)
        return -2;
    if (reinterpret_cast<uintptr_t>(points) % 4 != 0)
        return -1;
    const dim3 grid(static_cast<unsigned>((n + kEncThreads - 1) / kEncThreads), static_cast<unsigned>(groups)), block(kEncThreads);
    hipStream_t st = static_cast<hipStream_t>(stream);
    const uint16_t *d = static_cast<const uint16_t *>(data), *p = static_cast<const uint16_t *>(points);
    switch (P) {
    case 2: hipLaunchKernelGGL(sbvr_encoder_group_mse_kernel<2>, grid, block, 0, st, d, p, mse, G, n); break;
    case 4: hipLaunchKernelGGL(sbvr_encoder_group_mse_kernel<4>, grid, block, 0, st, d, p, mse, G, n); break;
    case 8: hipLaunchKernelGGL(sbvr_encoder_group_mse_kernel<8>, grid, block, 0, st, d, p, mse, G, n); break;
    case 16: hipLaunchKernelGGL(sbvr_encoder_group_mse_kernel<16>, grid, block, 0, st, d, p, mse, G, n); break;
    case 32: hipLaunchKernelGGL(sbvr_encoder_group_mse_kernel<32>, grid, block, 0, st, d, p, mse, G, n); break;
    case 64: hipLaunchKernelGGL(sbvr_encoder_group_mse_kernel<64>, grid, block, 0, st, d, p, mse, G, n); break;
    case 128: hipLaunchKernelGGL(sbvr_encoder_group_mse_kernel<128>, grid, block, 0, st, d, p, mse, G, n); break;
    default: hipLaunchKernelGGL(sbvr_encoder_group_mse_kernel<256>, grid, block, 0, st, d, p, mse, G, n); break;
    }
    return hipGetLastError() == hipSuccess ? 0 : -3;
}

int sbvr_hip_encoder_candidates_f16(const void *data, int G, const void *base, int bases, const void *b, int bs, const void *s, int ss,
                                    const void *axes, int steps, int S, void *lines, float *mse, void *stream)
{
    if (!data || !base || !b || !s || !axes || !lines || !mse || G <= 0 || bases <= 0 || bs <= 0 || ss <= 0 || steps <= 0)
        return -1;
    if (S < 2 || S > 6 || G > kEncMaxG || G % 4 != 0)
        return -2;
    const long family = static_cast<long>(bases) * bs * ss;
    long grid_lines = 1;
    for (int q = 0; q < S && grid_lines <= (1L << 28); ++q)
        grid_lines *= steps;
    if (static_cast<double>(bases) * bs * ss > (1 << 28) || grid_lines > (1L << 28))
        return -2;
    const CandidateArgs a{static_cast<const uint16_t *>(data), static_cast<const uint16_t *>(base), static_cast<const uint16_t *>(b),
                          static_cast<const uint16_t *>(s), static_cast<const uint16_t *>(axes), static_cast<uint16_t *>(lines), mse,
                          bases, ss, steps, static_cast<int>(family), static_cast<int>(family + grid_lines), G};
    const dim3 grid(static_cast<unsigned>((a.n + kEncThreads - 1) / kEncThreads)), block(kEncThreads);
    hipStream_t st = static_cast<hipStream_t>(stream);
    switch (S) {
    case 2: hipLaunchKernelGGL(sbvr_encoder_candidates_kernel<2>, grid, block, 0, st, a); break;
    case 3: hipLaunchKernelGGL(sbvr_encoder_candidates_kernel<3>, grid, block, 0, st, a); break;
    case 4: hipLaunchKernelGGL(sbvr_encoder_candidates_kernel<4>, grid, block, 0, st, a); break;
    case 5: hipLaunchKernelGGL(sbvr_encoder_candidates_kernel<5>, grid, block, 0, st, a); break;
    default: hipLaunchKernelGGL(sbvr_encoder_candidates_kernel<6>, grid, block, 0, st, a); break;
    }
    return hipGetLastError() == hipSuccess ? 0 : -3;
}

size_t sbvr_hip_encoder_state_bytes(void) { return 2 * sizeof(EncoderState); }

int sbvr_hip_encoder_scales(int S, int G, int bases, int n_offsets, int axis_values)
{
    sbvr_hip_encoder_run space{};
    space.bases[0] = bases;
    space.n_offsets[0] = n_offsets;
    space.axis_values[0] = axis_values;
    return S >= 2 && S <= 6 && G > 0 && G <= kEncMaxG && G % 4 == 0 && bases > 0 && n_offsets > 0 && axis_values > 1 && run_lines(space, 0, S) ? kEncMaxScales : 0;
}

int sbvr_hip_encoder_rounds_f16(const sbvr_hip_encoder_run *run, int S, int lines, int slot, int rounds, void *stream)
{
    if (!run_ok(run) || lines <= 0 || slot < 0 || slot > 1 || rounds <= 0)
        return -1;
    if (S < 2 || S > 6 || run->G > kEncMaxG || run->G % 4 != 0 || !run_lines(*run, 0, S) || !run_lines(*run, 1, S))
        return -2;
    const unsigned grid = static_cast<unsigned>((lines + kEncThreads - 1) / kEncThreads);
    hipStream_t st = static_cast<hipStream_t>(stream);
    switch (S) {
    case 2: launch_rounds<2>(*run, grid, slot, rounds, st); break;
    case 3: launch_rounds<3>(*run, grid, slot, rounds, st); break;
    case 4: launch_rounds<4>(*run, grid, slot, rounds, st); break;
    case 5: launch_rounds<5>(*run, grid, slot, rounds, st); break;
    default: launch_rounds<6>(*run, grid, slot, rounds, st); break;
    }
    return hipGetLastError() == hipSuccess ? 0 : -3;
}

int sbvr_hip_encoder_selectors_f16(const sbvr_hip_encoder_run *run, int S, int first, int groups, void *stream)
{
    if (!run_ok(run) || first < 0 || groups <= 0 || first + groups > run->groups)
        return -1;
    if (S < 2 || S > 6 || run->G > kEncMaxG)
        return -2;
    hipStream_t st = static_cast<hipStream_t>(stream);
    switch (S) {
    case 2: launch_selectors<2>(*run, first, groups, st); break;
    case 3: launch_selectors<3>(*run, first, groups, st); break;
    case 4: launch_selectors<4>(*run, first, groups, st); break;
    case 5: launch_selectors<5>(*run, first, groups, st); break;
    default: launch_selectors<6>(*run, first, groups, st); break;
    }
    return hipGetLastError() == hipSuccess ? 0 : -3;
}

int sbvr_hip_online_encode_f16(const void *x, const void *points, uint32_t *bvr, int M, int K, int G, int S, void *stream)
{
    if (!x || !points || !bvr || M <= 0 || K <= 0 || G <= 0 || S <= 0)
        return -1;
    if (S > 8 || G % 32 != 0 || K % G != 0 || M > 65535)
        return -2;
    const dim3 grid(static_cast<unsigned>((K + 63) / 64), static_cast<unsigned>((M + kOnlineRows - 1) / kOnlineRows)), block(64 * kOnlineWaves);
    hipLaunchKernelGGL((sbvr_online_encode_kernel<false, false>), grid, block, 0, static_cast<hipStream_t>(stream), static_cast<const uint16_t *>(x),
                       static_cast<const uint16_t *>(points), bvr, nullptr, 0, M, K, G, S, nullptr, nullptr);
    return hipGetLastError() == hipSuccess ? 0 : -3;
}

int sbvr_hip_online_encode_lines_f16(const void *x, const void *lines, uint32_t *bvr, void *idx, int idx_bytes, int M, int K, int G,
                                     int S, void *stream)
{
    if (!x || !lines || !bvr || !idx || M <= 0 || K <= 0 || G <= 0 || S <= 0 || (idx_bytes != 1 && idx_bytes != 2))
        return -1;
    if (S > 8 || G % 32 != 0 || K % G != 0 || M > 65535 || (idx_bytes == 1 && K / G > 256) || K / G > 65536)
        return -2;
    const dim3 grid(static_cast<unsigned>((K + 63) / 64), static_cast<unsigned>((M + kOnlineRows - 1) / kOnlineRows)), block(64 * kOnlineWaves);
    hipLaunchKernelGGL((sbvr_online_encode_kernel<true, false>), grid, block, 0, static_cast<hipStream_t>(stream), static_cast<const uint16_t *>(x),
                       static_cast<const uint16_t *>(lines), bvr, static_cast<uint8_t *>(idx), idx_bytes == 2 ? 1 : 0, M, K, G, S, nullptr, nullptr);
    return hipGetLastError() == hipSuccess ? 0 : -3;
}

size_t sbvr_hip_online_mm_T_scratch(const uint32_t *r_bvr, const void *r_cache, int M, int N, int K, int Sl, int Sr, int G)
{
    if (M <= 0 || N <= 0 || K <= 0 || Sl <= 0 || Sr <= 0 || G <= 0 || K % G != 0 || !online_product_ok(M, N, K, Sl, Sr, G, r_bvr, r_cache, device_cus()))
        return 0;
    const size_t image = static_cast<size_t>(K / 128) * ((M + 15) / 16) * 8192, planes = static_cast<size_t>(K / 32) * M * Sl * 4;
    return image + planes + static_cast<size_t>(K / G) * sizeof(float);
}

int sbvr_hip_online_mm_T(const void *x, const void *lines, const uint32_t *r_bvr, const void *r_idx, int r_idx_bytes, const void *r_cache,
                         const void *bias, void *out, int M, int N, int K, int Sl, int Sr, int G, int Lr, void *scratch,
                         size_t scratch_bytes, void *stream)
{
    if (!x || !lines || !r_bvr || !r_idx || !r_cache || !out || !scratch || M <= 0 || N <= 0 || K <= 0 || Sl <= 0 || Sr <= 0 || G <= 0 || Lr <= 0 ||
        (r_idx_bytes != 1 && r_idx_bytes != 2))
        return -1;
    const size_t need = sbvr_hip_online_mm_T_scratch(r_bvr, r_cache, M, N, K, Sl, Sr, G);
    if (!need || scratch_bytes < need || reinterpret_cast<uintptr_t>(scratch) % 16 != 0 || K / G > 65536)
        return -2;
    hipStream_t st = static_cast<hipStream_t>(stream);
    uint8_t *const at = static_cast<uint8_t *>(scratch);
    const size_t image = static_cast<size_t>(K / 128) * ((M + 15) / 16) * 8192, planes = static_cast<size_t>(K / 32) * M * Sl * 4;
    uint32_t *const bvr = reinterpret_cast<uint32_t *>(at + image);
    float *const scales = reinterpret_cast<float *>(at + image + planes);
    const dim3 grid(static_cast<unsigned>((K + 63) / 64), static_cast<unsigned>((M + kOnlineRows - 1) / kOnlineRows)), block(64 * kOnlineWaves);
    hipLaunchKernelGGL((sbvr_online_encode_kernel<true, true>), grid, block, 0, st, static_cast<const uint16_t *>(x), static_cast<const uint16_t *>(lines),
                       bvr, nullptr, 0, M, K, G, Sl, reinterpret_cast<uint32_t *>(at), scales);
    if (hipGetLastError() != hipSuccess)
        return -3;
    OnlineArgs a{};
    a.l_bvr = bvr;
    a.lines = static_cast<const uint16_t *>(lines);
    a.r_bvr = r_bvr;
    a.r_idx = r_idx;
    a.r_cache = static_cast<const uint16_t *>(r_cache);
    a.bias = static_cast<const uint16_t *>(bias);
    a.out = static_cast<uint16_t *>(out);
    a.image = reinterpret_cast<const v4u_image *>(at);
    a.scales = scales;
    a.M = M; a.N = N; a.K = K; a.Sl = Sl; a.Lr = Lr;
    a.r_idx16 = r_idx_bytes == 2;
    return launch_online_product(Sr, G, a, device_cus(), st) == hipSuccess ? 0 : -3;
}

int sbvr_hip_decode_weight(const uint32_t *bvr, const void *idx, int idx_bytes, const void *cache, void *out, int out_type, int N, int K,
                           int k_out, int S, int G, int L, void *stream)
{
    if (!bvr || !idx || !cache || !out || N <= 0 || K <= 0 || S <= 0 || G <= 0 || L <= 0 || k_out <= 0 || k_out > K ||
        (idx_bytes != 1 && idx_bytes != 2) || out_type < kOutF16 || out_type > kOutF32)
        return -1;
    const int words = K / 32;
    const long gy = (static_cast<long>(words) + 8 * kDecWaves - 1) / (8 * kDecWaves);
    if (G % 32 != 0 || K % G != 0 || gy > 65535)
        return -2;
    const size_t row_bytes = static_cast<size_t>(k_out) * (out_type == kOutF32 ? 4 : 2);
    DecodeArgs a{bvr, static_cast<const uint8_t *>(idx), static_cast<const uint16_t *>(cache), out, N, words, S, G / 32, L,
                 idx_bytes == 2 ? 1 : 0, k_out, row_bytes % 16 == 0 && reinterpret_cast<uintptr_t>(out) % 16 == 0 ? 1 : 0};
    const dim3 grid(static_cast<unsigned>((N + 7) / 8), static_cast<unsigned>(gy));
    const bool aligned = reinterpret_cast<uintptr_t>(bvr) % 16 == 0 && reinterpret_cast<uintptr_t>(cache) % 16 == 0;
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (aligned && S == 4)
        launch_decode<4>(out_type, grid, st, a);
    else if (aligned && S == 3)
        launch_decode<3>(out_type, grid, st, a);
    else if (aligned && S == 2)
        launch_decode<2>(out_type, grid, st, a);
    else if (aligned && S == 6)
        launch_decode<6>(out_type, grid, st, a);
    else if (aligned && S == 8)
        launch_decode<8>(out_type, grid, st, a);
    else
        launch_decode<0>(out_type, grid, st, a);
    return hipGetLastError() == hipSuccess ? 0 : -3;
}

}  // extern "C"
