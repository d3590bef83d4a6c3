// Both operands SBVR-encoded, any number of left rows (libsbvr_hip.so, gfx950): the reference's product
//   out[m, n] = sum_g sum_{l, r} popcount_g(L_l & R_r) a_l b_r      (sbvr_kernel.cu:462-562, sbvr_kernel.cpp:251-399)
// with the popcounts coming out of the matrix cores.
#include "sbvr_internal.h"
#include "sbvr_device.h"

namespace {

constexpr int kMmSub = 128;          // elements of K per MFMA

// A workgroup owns 16 columns and up to 16 * RT (left row, plane) pairs; its W waves take the sub-groups of 128
// elements of K in turn and meet in LDS.  Per sub-group a lane holds one plane word of its column and plane r and one
// word of each of its RT left rows, and v_mfma_f32_16x16x128_f8f6f4 with both operands fp4 multiplies the raw bits:
// nibble q of dword t carries bit 4q + t, as 0.5, 1, 2, 2 on the right and as 2, 1, 0.5, 0.5 on the left, so a
// product is 1 or 0 and the sums are the popcounts, exact integers in fp32.  A left row's planes are rows of their
// own ((K / 32, M, Sl) is (K / 32, M * Sl) as it lies), so any number of planes on that side takes the same code.
// Coefficients in fp32: those of the column per lane (its line, gathered one sub-group ahead), those of the left
// rows from a small LDS table that the wave fills for itself.
// Bound by the vector ALU: per 16 x 16 x 128 block and SR right planes 4 SR + 4 FMAs a lane, 7 operations to make the
// left operand, against 16 clocks per MFMA; with few rows by the latency of the loads in front of it.  (Where the
// one-thread-per-output kernel took 727 us, 16 rows of 8 planes x 4096 columns x 4096 with 4 right planes, it takes 9.8;
// 4 rows of 4 planes 4.7 us where the popcount kernel took 9.3.)
template <int SR, int RT, int W>
__global__ void __launch_bounds__(64 * W)
sbvr_mm_T_mfma_kernel(const MmArgs a)
{
    constexpr int R = 16 * RT;                       // (left row, plane) pairs of a workgroup
    constexpr int CW = (SR + 1) / 2;
    constexpr int PS = SR <= 4 ? SR : SR / 2, PH = SR / PS;     // planes of a step, steps per row tile
    constexpr int NL = (R + 63) / 64;                // left coefficients a lane fetches per sub-group
    __shared__ __align__(16) float red[W * R * 16];  // the partial results; before that the waves' coefficients
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int col = lane & 15, blk = lane >> 4;
    const int M = a.M, N = a.N, Sl = a.Sl;
    const int n = blockIdx.x * 16 + col, n_ld = min(n, N - 1);
    const int m0 = blockIdx.y * a.m_per_wg, m_cnt = min(a.m_per_wg, M - m0);
    const int rows = m_cnt * Sl, row0 = m0 * Sl, rows_all = M * Sl;
    const int nsub = a.K / kMmSub;
    float *const ca = red + wave * R;                // this wave's left coefficients

    // the left coefficients this lane fetches: pair p = lane + 64 i is plane p % Sl of left row p / Sl
    int lm[NL], lp[NL];
#pragma unroll
    for (int i = 0; i < NL; ++i) {
        const int p = min(lane + 64 * i, rows - 1);
        lm[i] = m0 + p / Sl;
        lp[i] = p % Sl;
    }

    struct Stage {
        Planes<SR> w;
        uint32_t aw[RT];
        int r_lo, r_hi, l_lo[NL], l_hi[NL];          // line indices, as loaded (one or two bytes)
        uint32_t rc[CW];
        uint16_t lc[NL];
    };
    auto load = [&](int sg, Stage &s) __attribute__((always_inline)) {
        const size_t word = static_cast<size_t>(4 * sg + blk);
        s.w = load_planes<SR>(a.r_bvr + (word * N + n_ld) * SR);
#pragma unroll
        for (int t = 0; t < RT; ++t)
            s.aw[t] = a.l_bvr[word * rows_all + min(row0 + 16 * t + col, rows_all - 1)];
        const int g = sg / a.spg;
        const uint8_t *rb = static_cast<const uint8_t *>(a.r_idx), *lb = static_cast<const uint8_t *>(a.l_idx);
        const size_t rat = (static_cast<size_t>(g) * N + n_ld) << a.r_idx16;
        s.r_lo = rb[rat];
        s.r_hi = rb[rat + a.r_idx16];
#pragma unroll
        for (int i = 0; i < NL; ++i) {
            const size_t lat = (static_cast<size_t>(g) * M + lm[i]) << a.l_idx16;
            s.l_lo[i] = lb[lat];
            s.l_hi[i] = lb[lat + a.l_idx16];
        }
    };
    auto gather = [&](Stage &s) __attribute__((always_inline)) {
        const int rline = min(a.r_idx16 ? s.r_lo | (s.r_hi << 8) : s.r_lo, a.Lr - 1);
        load_line_words<SR>(a.r_cache + static_cast<size_t>(rline) * SR, s.rc);
#pragma unroll
        for (int i = 0; i < NL; ++i) {
            const int lline = min(a.l_idx16 ? s.l_lo[i] | (s.l_hi[i] << 8) : s.l_lo[i], a.Ll - 1);
            s.lc[i] = a.l_cache[static_cast<size_t>(lline) * Sl + lp[i]];
        }
    };

    v4f y[RT];
#pragma unroll
    for (int t = 0; t < RT; ++t)
        y[t] = v4f{0.f, 0.f, 0.f, 0.f};
    auto compute = [&](const Stage &s) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NL; ++i)
            if (NL == 1 ? lane < R : true)
                ca[lane + 64 * i] = h2f(s.lc[i]);
        __builtin_amdgcn_wave_barrier();
        v8i B[SR];
        float c[SR];
#pragma unroll
        for (int j = 0; j < SR; ++j) {
            const uint32_t w = s.w.w[j];
            B[j] = v8i{static_cast<int>(w & 0x11111111u), static_cast<int>(w & 0x22222222u), static_cast<int>(w & 0x44444444u),
                       static_cast<int>((w >> 1) & 0x44444444u), 0, 0, 0, 0};
            c[j] = h2f(static_cast<uint16_t>(j & 1 ? s.rc[j / 2] >> 16 : s.rc[j / 2] & 0xffffu));
        }
        // A step is up to 4 planes of one row tile: its MFMAs are issued together, and the results of the step before
        // are multiplied with their coefficients while they run (left to itself the compiler lets every MFMA's
        // consumers wait for it before it issues the next one: 118 us against 110 for 64 rows of 8 planes x 14336 x 4096 with 8 row tiles)
        v4f D[2][PS];
        v4f sum = v4f{0.f, 0.f, 0.f, 0.f};
        auto consume = [&](int step) __attribute__((always_inline)) {
            const int t = step / PH, ph = step % PH;
#pragma unroll
            for (int j = 0; j < PS; ++j)
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    sum[i] = ph == 0 && j == 0 ? D[step & 1][j][i] * c[0] : fmaf(D[step & 1][j][i], c[ph * PS + j], sum[i]);
            if (ph == PH - 1) {
                const v4f la = *reinterpret_cast<const v4f *>(ca + 16 * t + 4 * blk);
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    y[t][i] = fmaf(la[i], sum[i], y[t][i]);
            }
        };
        v8i A;
#pragma unroll
        for (int step = 0; step < RT * PH; ++step) {
            if (step % PH == 0) {
                const uint32_t w = s.aw[step / PH];
                A = v8i{static_cast<int>((w << 2) & 0x44444444u), static_cast<int>(w & 0x22222222u),
                        static_cast<int>((w >> 2) & 0x11111111u), static_cast<int>((w >> 3) & 0x11111111u), 0, 0, 0, 0};
            }
#pragma unroll
            for (int j = 0; j < PS; ++j)
                D[step & 1][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(A, B[(step % PH) * PS + j], v4f{0.f, 0.f, 0.f, 0.f},
                                                                                  4, 4, 0, 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            if (step > 0)
                consume(step - 1);
            __builtin_amdgcn_sched_barrier(0);
        }
        consume(RT * PH - 1);
        __builtin_amdgcn_wave_barrier();
    };

    // (two register sets; a sub-group past the end repeats the last one and is not computed)
    Stage s0, s1;
    if (wave < nsub) {                               // wave-uniform
        load(wave, s0);
        gather(s0);
        for (int sg = wave; sg < nsub; sg += 2 * W) {
            load(min(sg + W, nsub - 1), s1);
            __builtin_amdgcn_sched_barrier(0);
            compute(s0);
            gather(s1);
            if (sg + W >= nsub)
                break;
            load(min(sg + 2 * W, nsub - 1), s0);
            __builtin_amdgcn_sched_barrier(0);
            compute(s1);
            gather(s0);
        }
    }
    __syncthreads();                                 // (the coefficients' place is free now)

    // partial results: [wave][pair][column]
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i)
            red[(wave * R + 16 * t + 4 * blk + i) * 16 + col] = y[t][i];
    __syncthreads();
    for (int o = threadIdx.x; o < rows * 16; o += 64 * W) {     // over the waves, per (pair, column)
        float total = 0.f;
#pragma unroll
        for (int w = 0; w < W; ++w)
            total += red[w * R * 16 + o];
        red[o] = total;                              // (this thread's own slot of wave 0)
    }
    __syncthreads();
    for (int o = threadIdx.x; o < m_cnt * 16; o += 64 * W) {    // over the planes of a left row
        const int mm = o >> 4, cc = o & 15, nn = blockIdx.x * 16 + cc;
        float total = 0.f;
        for (int l = 0; l < Sl; ++l)
            total += red[(mm * Sl + l) * 16 + cc];
        if (nn < N) {
            uint16_t v = f2h(total);
            if (a.bias)
                v = hadd(v, a.bias[nn]);
            a.out[static_cast<size_t>(m0 + mm) * N + nn] = v;
        }
    }
}

// ------------------------------------------------------- activations encoded on the fly, more than a few of them
//
// The left operand of that product is a dense matrix a_hat[m, k] = sum_l a_l(group) L_l[m, k]: its coefficient line belongs to
// the group, not to the row, so the launch that encodes the activations leaves it as fp16 numbers too (two parts, in the
// order of the MFMA's A operand: OnlineArgs), and the right planes' bits meet it as fp16 numbers: a word of this layout holds
// 32 k of one column, shifted it has the pair (k = i, i + 16) at the same exponent bit of either half, and one `and` leaves a ready
// dword of the B operand of v_mfma_f32_16x16x32_f16, a power of two each that the activations carry the inverse of.  So 16 left
// rows are one row tile of 8 MFMAs a plane and 128 k, where their planes are 8 tiles above whose sums each want a
// multiplication: 19 operations a plane word and 12 a plane's sums, against 7 + 20 for each of the 8 tiles.  A workgroup owns 16
// columns and 16 RT rows; its W waves take the sub-groups of 128 k in turn and meet in LDS.  Bound by latency, and by the
// image's way through the L1 (8 KiB a sub-group and row tile, for every 16 columns).
// As exact as the planes' own product, in front of the output's rounding and over the RMS output: 0.37 to 0.51e-7 where that has
// 0.8 to 2.0e-7, with input coefficients of one sign 0.39 to 0.48e-7 and 0.49 to 0.76e-7 (12 to 64 rows, 2 to 8 planes, K 128 to 14336).
// Each of these matters: powers of two that are normal numbers (the bits where they lie are subnormal ones, which the matrix cores
// line up by their least exponent: 25e-7); sums of the first parts, exact, and of the second ones apart, and differences of planes
// (in one sum 2e-7 with coefficients of one sign; 4 us of 30 less, 64 rows x 4096, K 4096); the sub-groups' sums added up in 64
// bits (in 32: up to 0.9e-7, and as fast).
template <int SR, int RT, int W>
__global__ void __launch_bounds__(64 * W)
sbvr_online_product_kernel(const OnlineArgs a)
{
    constexpr int CW = (SR + 1) / 2;
    __shared__ __align__(16) double red[W * RT * 256];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int col = lane & 15, blk = lane >> 4;
    const int N = a.N, nsub = a.K / kMmSub;
    const int n = blockIdx.x * 16 + col, n_ld = min(n, N - 1);
    const int tiles = (a.M + 15) / 16, t0 = blockIdx.y * RT;         // row tiles of the image, and the first of this workgroup's

    struct Stage {
        Planes<SR> w;
        int lo, hi;
        uint32_t c[CW];
        float scale;
    };
    auto load = [&](int sg, Stage &s) __attribute__((always_inline)) {
        s.w = load_planes<SR>(a.r_bvr + (static_cast<size_t>(4 * sg + blk) * N + n_ld) * SR);
        const uint8_t *rb = static_cast<const uint8_t *>(a.r_idx);
        const size_t at = (static_cast<size_t>(sg / a.spg) * N + n_ld) << a.r_idx16;
        s.lo = rb[at];
        s.hi = rb[at + a.r_idx16];
        s.scale = a.scales[sg / a.spg];
    };
    auto gather = [&](Stage &s) __attribute__((always_inline)) {
        const int line = min(a.r_idx16 ? s.lo | (s.hi << 8) : s.lo, a.Lr - 1);
        load_line_words<SR>(a.r_cache + static_cast<size_t>(line) * SR, s.c);
    };
    auto coefficient = [&](const Stage &s, int j) __attribute__((always_inline)) -> float {
        return h2f(static_cast<uint16_t>(j & 1 ? s.c[j / 2] >> 16 : s.c[j / 2] & 0xffffu));
    };
    double y[RT][4] = {};
    // Whether a coefficient of this lane's column is not finite.
    auto not_finite_line = [&](const Stage &s) __attribute__((always_inline)) -> bool {
        bool bad = false;
#pragma unroll
        for (int j = 0; j < SR; ++j)
            bad = bad || !(fabsf(coefficient(s, j)) < INFINITY);
        return bad;
    };
    // Such a column's sub-group by popcounts, as sbvr_mm_T_mfma_kernel has them, a left plane of all rows at a time: a left plane
    // that shares no bit with that coefficient's plane makes NaN of the output (0 times infinity).
    auto plane_by_plane = [&](int sg, const Stage &s, bool mine) __attribute__((always_inline)) {
#pragma unroll 1
        for (int l = 0; l < a.Sl; ++l) {
            const float c = h2f(a.lines[static_cast<size_t>(sg / a.spg) * a.Sl + l]);
#pragma unroll
            for (int t = 0; t < RT; ++t) {
                const uint32_t left = a.l_bvr[(static_cast<size_t>(4 * sg + blk) * a.M + min((t0 + t) * 16 + col, a.M - 1)) * a.Sl + l];
                const v8i A = {static_cast<int>((left << 2) & 0x44444444u), static_cast<int>(left & 0x22222222u),
                               static_cast<int>((left >> 2) & 0x11111111u), static_cast<int>((left >> 3) & 0x11111111u), 0, 0, 0, 0};
                v4f sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int j = 0; j < SR; ++j) {
                    const uint32_t w = s.w.w[j];
                    const v8i B = {static_cast<int>(w & 0x11111111u), static_cast<int>(w & 0x22222222u), static_cast<int>(w & 0x44444444u),
                                   static_cast<int>((w >> 1) & 0x44444444u), 0, 0, 0, 0};
                    const v4f count = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(A, B, v4f{0.f, 0.f, 0.f, 0.f}, 4, 4, 0, 0, 0, 0);
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        sum[i] = fmaf(count[i], coefficient(s, j), sum[i]);
                }
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    y[t][i] += mine ? static_cast<double>(c * sum[i]) : 0.;
            }
        }
    };
    bool any_bad = false;
    auto compute = [&](int sg, const Stage &s) __attribute__((always_inline)) {
        // (asked for a sub-group ahead, in 32 registers more, the image's operands cost 1 us of 6.5)
        const v4u *const image = a.image + static_cast<size_t>(sg) * tiles * 512 + lane;
        v4f D[2][SR][RT];                                            // of the activations' first parts and of the second ones
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            v4u A[RT][2];
#pragma unroll
            for (int t = 0; t < RT; ++t)
#pragma unroll
                for (int part = 0; part < 2; ++part)                 // (a tile past the last one repeats it)
                    A[t][part] = image[(min(t0 + t, tiles - 1) * 4 + u) * 128 + part * 64];
#pragma unroll
            for (int j = 0; j < SR; ++j) {
                const uint32_t w = s.w.w[j];
                v4u B;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int i = 4 * u + e;
                    B[e] = (i < 5 ? w << 10 : (i < 10 ? w << 5 : (i < 15 ? w : w >> 1))) & (0x04000400u << online_bit(i));
                }
#pragma unroll
                for (int part = 0; part < 2; ++part)
#pragma unroll
                    for (int t = 0; t < RT; ++t)
                        D[part][j][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8h, A[t][part]), __builtin_bit_cast(v8h, B),
                                                                               u == 0 ? v4f{0.f, 0.f, 0.f, 0.f} : D[part][j][t], 0, 0, 0);
            }
        }
        // A column's coefficients may almost cancel where its planes' sums are large and alike (activations of one sign).  The first
        // parts' sums are exact, so what two planes' differ by is: that meets the coefficients, and the first plane's sum theirs.
        // (a line that is not finite counts as zeros here: its sub-groups follow at the end, without a branch in this loop, which
        // took 0.5 us of 12)
        const bool bad = not_finite_line(s);
        any_bad = any_bad || bad;
        float c[SR], all = 0.f;
#pragma unroll
        for (int j = 0; j < SR; ++j) {
            c[j] = bad ? 0.f : coefficient(s, j);
            all += c[j];
        }
#pragma unroll
        for (int t = 0; t < RT; ++t)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                float sum = D[1][0][t][i] * c[0];
#pragma unroll
                for (int j = 1; j < SR; ++j)
                    sum = fmaf(D[1][j][t][i], c[j], sum);
#pragma unroll
                for (int j = 1; j < SR; ++j)
                    sum = fmaf(D[0][j][t][i] - D[0][0][t][i], c[j], sum);
                y[t][i] += static_cast<double>(fmaf(D[0][0][t][i], all, sum) * s.scale);
            }
    };
    if (wave < nsub) {                                               // wave-uniform
        Stage now, next;
        load(wave, now);
        gather(now);
        for (int sg = wave; sg < nsub; sg += W) {
            load(min(sg + W, nsub - 1), next);
            __builtin_amdgcn_sched_barrier(0);
            compute(sg, now);
            gather(next);
            now = next;
        }
        if (__any(any_bad))
#pragma unroll 1
            for (int sg = wave; sg < nsub; sg += W) {
                load(sg, now);
                gather(now);
                const bool bad = not_finite_line(now);
                if (__any(bad))
                    plane_by_plane(sg, now, bad);
            }
    }
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i)
            red[(wave * RT + t) * 256 + (4 * blk + i) * 16 + col] = y[t][i];
    __syncthreads();
    for (int o = threadIdx.x; o < RT * 256; o += 64 * W) {
        const int m = t0 * 16 + (o >> 4), nn = blockIdx.x * 16 + (o & 15);
        if (m >= a.M || nn >= N)
            continue;
        double total = 0.;
#pragma unroll
        for (int w = 0; w < W; ++w)
            total += red[w * RT * 256 + o];
        uint16_t v = f2h(static_cast<float>(total));
        if (a.bias)
            v = hadd(v, a.bias[nn]);
        a.out[static_cast<size_t>(m) * N + nn] = v;
    }
}

template <int SR, int RT, int W>
hipError_t launch_online_inst(const OnlineArgs &a, hipStream_t st)
{
    const dim3 grid(static_cast<unsigned>((a.N + 15) / 16), static_cast<unsigned>((a.M + 16 * RT - 1) / (16 * RT)));
    hipLaunchKernelGGL((sbvr_online_product_kernel<SR, RT, W>), grid, dim3(64 * W), 0, st, a);
    return hipGetLastError();
}

// (two row tiles of more planes: 130 to 248 registers; 8 planes of a 16-wave workgroup: more than its 128)
template <int SR>
hipError_t launch_online(int RT, int W, const OnlineArgs &a, hipStream_t st)
{
    if constexpr (SR == 2)
        if (RT == 2)
            return W == 16 ? launch_online_inst<SR, 2, 16>(a, st) : launch_online_inst<SR, 2, 8>(a, st);
    if constexpr (SR <= 6)
        if (W == 16)
            return launch_online_inst<SR, 1, 16>(a, st);
    return launch_online_inst<SR, 1, 8>(a, st);
}

template <int SR>
hipError_t launch_rt(int RT, int W, const MmArgs &a, hipStream_t st)
{
    const dim3 grid(static_cast<unsigned>((a.N + 15) / 16), static_cast<unsigned>((a.M + a.m_per_wg - 1) / a.m_per_wg)), block(64 * W);
    if (RT == 4)
        hipLaunchKernelGGL((sbvr_mm_T_mfma_kernel<SR, 4, 8>), grid, block, 0, st, a);
    else if (RT == 2 && W == 16)
        hipLaunchKernelGGL((sbvr_mm_T_mfma_kernel<SR, 2, 16>), grid, block, 0, st, a);
    else if (RT == 2)
        hipLaunchKernelGGL((sbvr_mm_T_mfma_kernel<SR, 2, 8>), grid, block, 0, st, a);
    else if (W == 16)
        hipLaunchKernelGGL((sbvr_mm_T_mfma_kernel<SR, 1, 16>), grid, block, 0, st, a);
    else
        hipLaunchKernelGGL((sbvr_mm_T_mfma_kernel<SR, 1, 8>), grid, block, 0, st, a);
    return hipGetLastError();
}

}  // namespace

// (at most 65535 blocks of left rows, of 64 (row, plane) pairs each where there are that many: the grid's y)
bool mm_T_mfma_ok(int M, int N, int K, int Sl, int Sr, int G, const void *r_bvr, const void *r_cache)
{
    if (Sl > 16 || (static_cast<long>(M) + 64 / Sl - 1) / (64 / Sl) > 65535)
        return false;
    return K % kMmSub == 0 && G % kMmSub == 0 && (Sr == 2 || Sr == 3 || Sr == 4 || Sr == 6 || Sr == 8) &&
           static_cast<double>(M) * Sl * (K / 32) < 2147483648.0 && static_cast<double>(N) * Sr * (K / 32) < 2147483648.0 &&
           reinterpret_cast<uintptr_t>(r_bvr) % 16 == 0 && reinterpret_cast<uintptr_t>(r_cache) % 16 == 0;
}

hipError_t launch_mm_T_mfma(int Sr, int G, MmArgs a, int cus, hipStream_t st)
{
    a.spg = G / kMmSub;
    // The fewest row tiles that hold all (left row, plane) pairs, up to 4; fewer again while the workgroups leave a
    // quarter of the CUs without one (every workgroup of a column block reads its plane words again, out of the L2).
    // Sixteen waves where that gives a CU about one workgroup, eight where there are two and more.  us by (row tiles,
    // waves), 4 right planes: 16 rows of 8 planes, 4096 x 4096: (4, 8) 9.7, (8, 8) 9.8, (4, 16) 11.7, (2, 16) 15.4;
    // 64 rows of 8 planes, 14336 x 4096: (4, 8) 89.5 to 99, (8, 8) 110, (4, 16) 133; 32 rows of 8, 512 x 14336: (2, 16) 10.0,
    // (1, 16) 12.2, (4, 16) 13.5; 4 rows of 4, 4096 x 4096: (1, 16) 4.9, (1, 8) 5.3, (1, 4) 6.8.
    const int rows = a.M * a.Sl, cols = (a.N + 15) / 16;
    int RT = rows <= 16 ? 1 : (rows <= 32 ? 2 : 4);
    auto m_per_wg = [&](int rt) { return 16 * rt / a.Sl; };
    auto wgs = [&](int rt) { return static_cast<long>(cols) * ((a.M + m_per_wg(rt) - 1) / m_per_wg(rt)); };
    while (RT > 1 && m_per_wg(RT / 2) >= 1 && wgs(RT) * 4 < 3L * cus)
        RT /= 2;
    a.m_per_wg = m_per_wg(RT);
    const int W = RT == 4 || wgs(RT) >= 2L * cus ? 8 : 16;
    switch (Sr) {
    case 2: return launch_rt<2>(RT, W, a, st);
    case 3: return launch_rt<3>(RT, W, a, st);
    case 4: return launch_rt<4>(RT, W, a, st);
    case 6: return launch_rt<6>(RT, W, a, st);
    default: return launch_rt<8>(RT, W, a, st);
    }
}

// Where that way is the faster one: more than 4 left planes, workgroups for three quarters of the CUs, and row tiles for whose
// rows the planes' launch takes a third more workgroups, of up to 64 (row, plane) pairs.  us a call (both launches), planes and
// this, 8 left and 4 right planes: 9 rows x 4096, K 4096 13.7 and 11.9; 64 rows 36.2 and 29.9; 32 x 14336, K 4096 52.4 and
// 39.6; 48 x 1024, K 14336 43.2 and 38.8; 2048 x 4096, K 4096 973 and 717; but (too few workgroups) 16 x 1024, K 14336 17.4 and
// 23.0; 64 x 512, K 4096 15.8 and 17.5; (4 left planes) 32 x 4096, K 4096 12.2 and 12.9; (6 left planes: two workgroups, two tiles)
// 20 rows 13.0 and 15.5.  At four workgroups to three tiles it is 0.8 to 1.35 times as fast, the mean of 140 shapes 1.  Images (4
// bytes an activation, in memory of the call's own) up to the largest measured: 2048 x 1024, K 14336 1287 us and 1150.
constexpr double kOnlineImageMost = 128 << 20;
bool online_product_ok(int M, int N, int K, int Sl, int Sr, int G, const void *r_bvr, const void *r_cache, int cus)
{
    const long tiles = (static_cast<long>(M) + 15) / 16;
    return mm_T_mfma_ok(M, N, K, Sl, Sr, G, r_bvr, r_cache) && Sl > 4 && Sl <= 8 && M <= 4096 &&
           3 * ((static_cast<long>(M) + 64 / Sl - 1) / (64 / Sl)) >= 4 * tiles && static_cast<long>((N + 15) / 16) * tiles * 4 >= 3L * cus &&
           static_cast<double>(tiles) * (K / kMmSub) * 8192 <= kOnlineImageMost;
}

// Two row tiles share a plane word's operands where the registers hold both, with 2 planes.  (us a call, one and two, 64 rows x 4096, K
// 4096: 4 planes 29.5 and 30.7; 33 rows, 3 planes 21.1 and 24.8.)
hipError_t launch_online_product(int Sr, int G, OnlineArgs a, int cus, hipStream_t st)
{
    a.spg = G / kMmSub;
    const int tiles = (a.M + 15) / 16, cols = (a.N + 15) / 16;
    const int RT = Sr == 2 && tiles > 1 && static_cast<long>(cols) * ((tiles + 1) / 2) * 4 >= 3L * cus ? 2 : 1;
    const int W = static_cast<long>(cols) * ((tiles + RT - 1) / RT) >= 2L * cus ? 8 : 16;
    switch (Sr) {
    case 2: return launch_online<2>(RT, W, a, st);
    case 3: return launch_online<3>(RT, W, a, st);
    case 4: return launch_online<4>(RT, W, a, st);
    case 6: return launch_online<6>(RT, W, a, st);
    default: return launch_online<8>(RT, W, a, st);
    }
}
