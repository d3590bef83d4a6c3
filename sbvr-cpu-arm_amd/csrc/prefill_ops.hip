// Prefill with five to eight row blocks a workgroup: the dense contraction of sbvr_gemm_lut_kernel (sbvr_hip.hip) as one
// instruction stream in which the decode runs between the MFMAs (libsbvr_hip.so, gfx950).
#include <mutex>
#include <type_traits>
#include <utility>
#include "sbvr_internal.h"
#include "sbvr_device.h"

namespace {

// f(0), f(1), ..., f(N - 1) with the index known to the compiler
template <int... I, typename F>
__device__ __forceinline__ void static_for_each(std::integer_sequence<int, I...>, F &&f)
{
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void static_for(F &&f)
{
    static_for_each(std::make_integer_sequence<int, N>{}, static_cast<F &&>(f));
}

// lut_build_tables (the same operations) in three pieces
template <int S>
struct TablePieces {
    float s[1 << S];
    v2h e[1 << (S - 1)];
    __device__ __forceinline__ void sums(const uint32_t (&c)[(S + 1) / 2])
    {
        float cf[S];
#pragma unroll
        for (int q = 0; q < S; ++q)
            cf[q] = h2f(static_cast<uint16_t>(q & 1 ? c[q / 2] >> 16 : c[q / 2] & 0xffffu));
        s[0] = 0.f;
#pragma unroll
        for (int q = 0; q < S; ++q)
#pragma unroll
            for (int i = 0; i < (1 << q); ++i)
                s[(1 << q) + i] = i == 0 ? cf[q] : s[i] + cf[q];
    }
    __device__ __forceinline__ void round()
    {
#pragma unroll
        for (int i = 0; i < (1 << (S - 1)); ++i) {
            e[i][0] = static_cast<_Float16>(s[2 * i]);
            e[i][1] = static_cast<_Float16>(s[2 * i + 1]);
        }
    }
    __device__ __forceinline__ void bytes(LutTables<S> &t)
    {
#pragma unroll
        for (int i = 0; i < LutTables<S>::TW; ++i) {
            const uint32_t e0 = __builtin_bit_cast(uint32_t, e[2 * i]), e1 = __builtin_bit_cast(uint32_t, e[2 * i + 1]);
            t.lo[i] = __builtin_amdgcn_perm(e1, e0, 0x06040200u);
            t.hi[i] = __builtin_amdgcn_perm(e1, e0, 0x07050301u);
        }
    }
};

typedef v4u __attribute__((aligned(2))) v4u_any;

constexpr int kPfWaves = 8, kPfBN = 256, kPfRow = 144;

// What a step does between its MFMAs, in units of 3 to 16 instructions, and behind which of its 4 RB MFMAs each unit
// stands: spread evenly by their instructions.
template <int S, int RB, bool kShare>
struct StepPlan {
    static constexpr int kLook = S <= 3 ? 1 : (S == 6 ? 2 : 3);                   // units of a look-up (8 look-ups of 4 weights a step)
    static constexpr int kStores = 4;                                             // activations of the next step to LDS
    static constexpr int kNib = kStores, kLoads = kNib + 4, kTabs = kLoads + 2;   // selectors, requests, tables
    static constexpr int kCoeffs = kTabs + 3, kLooks = kCoeffs + 1, kUnits = kLooks + 8 * kLook;
    static constexpr int cost(int u, bool odd)
    {
        if (u < kNib)
            return 5;
        if (u < kLoads)
            return S <= 4 ? (u == kNib ? 6 : 3) : (u == kNib ? 14 : 8);
        if (u < kTabs)
            return 4;
        if (u == kCoeffs)
            return kShare && !odd ? 0 : 8;
        if (u < kLooks) {
            if (S > 4)
                return !kShare || odd ? 16 : 0;
            if (!kShare)
                return S == 4 ? 13 : 6;
            return odd ? (u == kTabs ? 2 * S : 0) : (u == kTabs ? 0 : 2 * S + 1);
        }
        return S <= 3 ? 6 : (S == 4 ? 4 : ((u - kLooks) % kLook == 0 ? 6 : 8));
    }
    // the slots of an even and of an odd step: units first[odd][i] to first[odd][i + 1] - 1 stand behind MFMA i
    struct Slots {
        int first[2][4 * RB + 1] = {};
    };
    static constexpr Slots slots()
    {
        Slots s;
        for (int odd = 0; odd < 2; ++odd) {
            int all = 0, before = 0, u = 0;
            for (int v = 0; v < kUnits; ++v)
                all += cost(v, odd);
            for (int i = 0; i < 4 * RB; ++i) {
                s.first[odd][i] = u;
                while (u < kUnits && (2 * before + cost(u, odd)) * (4 * RB) < (2 * all + 1) * (i + 1))
                    before += cost(u++, odd);
            }
            s.first[odd][4 * RB] = kUnits;
        }
        return s;
    }
    static constexpr Slots kSlots = slots();
};

// The tiles, operands and decode are sbvr_gemm_lut_kernel's, and the results are its bit for bit.  There a step's decode and
// its MFMAs come in lumps, and a SIMD's two waves, kept together by the step's barrier, are in the same lump: a step of 8 row blocks
// takes 3500 clocks, 2048 of them MFMAs.  A SIMD hides up to six vector operations behind each MFMA of 32 clocks if they stand evenly
// between the MFMAs (a loop of one MFMA and 5 v_perm_b32, two waves: 34 clocks a turn; of 4 and 20: 44), so:
// * a step is laid out by hand, one MFMA, one operand read and one or two units of the rest in turn (StepPlan), fenced so that the
//   scheduler leaves them there: the operands of the next step are decoded, the activations of the next stored, the requests
//   for the one after sent between the MFMAs of this one;
// * activation tiles in three buffers, so that the barrier falls in the middle of a step and its successor's first operands
//   are read in front of it without a wait; an operand is read three MFMAs ahead, into four registers sets instead of 16;
// * addresses are uniform bases, moved on by selects, and 32-bit offsets: no vector arithmetic; no branch in the loop, behind which
//   the compiler would sink the units;
// * results (not split) go out through LDS, 16 bytes a lane: 128 stores a lane of 2 bytes took 14 us at the end of a launch.
// 2900 clocks a step of 8 row blocks and 4 planes.  What is left above the MFMAs: the LDS, whose 256 KiB of operand reads a step
// are 2048 clocks too, and the stores of the activations in between.  All CUs busy, the part runs at 1.5 to 1.6 GHz
// (2.4 with an eighth of them), whatever stands between the MFMAs.
template <int S, int RB, bool kShare>
__global__ void __launch_bounds__(64 * kPfWaves)
__attribute__((amdgpu_waves_per_eu(2, 4)))
sbvr_gemm_lut_pipelined_kernel(const GemmArgs a)
{
    static_assert(RB >= 5 && RB <= 8, "row blocks of a workgroup: 512 threads bring in 256 rows");
    using Plan = StepPlan<S, RB, kShare>;
    constexpr int kRing = 4, kAhead = kRing - 1;                    // operand registers, MFMAs from a read to its use
    constexpr int NQ = 4, kTile = 256 * kPfRow, CW = (S + 1) / 2;
    static_assert(Plan::kSlots.first[0][2 * RB - kAhead] >= Plan::kStores && Plan::kSlots.first[1][2 * RB - kAhead] >= Plan::kStores,
                  "kAhead reads behind the last store and in front of the barrier");
    extern __shared__ __align__(16) unsigned char psm[];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int N = a.N, K = a.K, M = a.M;
    const int j = lane & 31, h = lane >> 5;
    const int n0 = blockIdx.x * kPfBN, m0 = blockIdx.y * (32 * RB);
    const int n = n0 + 32 * wave + j, n_ld = min(n, N - 1);
    const int p0 = blockIdx.z * a.part_steps, p_last = min(p0 + a.part_steps, K / 64) - 1;      // this workgroup's steps (kShare: an even number)

    // bringing activations in: a thread takes word xw of row xr of a step
    const int xr = tid >> 1, xw = tid & 1;
    unsigned char *const xdst = psm + xr * kPfRow + xw * 64;
    const unsigned char *const xrd = psm + j * kPfRow + h * 64;      // + 32 rb rows, + 16 q

    // requests: bases of a step, moved on step by step (the last step again behind the end), and this lane's offsets
    const uint32_t x_at = (static_cast<uint32_t>(min(m0 + xr, M - 1)) * static_cast<uint32_t>(K) + 32 * xw) * 2u;
    const uint32_t w_at = static_cast<uint32_t>(h * N + n_ld) * (4u * S), i_at = static_cast<uint32_t>(n_ld) << a.idx16;
    const uint8_t *x_base = reinterpret_cast<const uint8_t *>(a.x + 64 * p0);
    const uint8_t *w_base = reinterpret_cast<const uint8_t *>(a.bvr + static_cast<size_t>(2 * p0) * N * S);
    const uint8_t *i_base = static_cast<const uint8_t *>(a.idx) + (static_cast<size_t>(p0 / a.steps_per_group) * N << a.idx16);
    const size_t w_step = static_cast<size_t>(2 * N) * (4 * S), i_step = static_cast<size_t>(N) << a.idx16;
    constexpr int kLineSteps = kShare ? 2 : 1;                       // steps that share a coefficient line
    int i_ip = p0, i_left = a.steps_per_group - p0 % a.steps_per_group;      // the step that i_base is of, and how many until the next group
    auto next_words = [&](int ip) __attribute__((always_inline)) {   // from step ip to ip + 1
        x_base += ip < p_last ? 128 : 0;
        w_base += ip < p_last ? w_step : 0;
    };
    auto next_line = [&]() __attribute__((always_inline)) {
        i_ip += kLineSteps;
        i_left -= kLineSteps;
        i_base += i_left == 0 && i_ip <= p_last ? i_step : 0;
        i_left += i_left == 0 ? a.steps_per_group : 0;
    };
    struct Line {
        int lo, hi;
    };
    auto load_line = [&]() __attribute__((always_inline)) -> Line { return Line{i_base[i_at], i_base[i_at + a.idx16]}; };
    Line line_of_next;
    uint32_t w[S], c[CW], x[16];                                     // x: dword 4 i + q: dword q of 16-byte chunk i
    auto load_coefficients = [&](const Line &line) __attribute__((always_inline)) {
        const int ln = min(a.idx16 ? line.lo | (line.hi << 8) : line.lo, a.L - 1);
        load_line_words<S>(a.cache + static_cast<size_t>(ln) * S, c);
    };
    auto load_words = [&]() __attribute__((always_inline)) {
        const Planes<S> pl = load_planes<S>(reinterpret_cast<const uint32_t *>(w_base + w_at));
#pragma unroll
        for (int q = 0; q < S; ++q)
            w[q] = pl.w[q];
    };
    auto load_x = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const v4u v = *reinterpret_cast<const v4u *>(x_base + x_at + 16 * i);
            x[4 * i] = v.x; x[4 * i + 1] = v.y; x[4 * i + 2] = v.z; x[4 * i + 3] = v.w;
        }
    };
    // the 32 elements of a (row, word) in the order of the MFMAs' A operands (sbvr_gemm_lut_kernel), operand q
    auto store_x = [&](int tile, int q) __attribute__((always_inline)) {
        v4u aw;
        aw.x = __builtin_amdgcn_perm(x[4 + q], x[q], 0x05040100u);
        aw.y = __builtin_amdgcn_perm(x[12 + q], x[8 + q], 0x05040100u);
        aw.z = __builtin_amdgcn_perm(x[4 + q], x[q], 0x07060302u);
        aw.w = __builtin_amdgcn_perm(x[12 + q], x[8 + q], 0x07060302u);
        *reinterpret_cast<v4u *>(xdst + tile + 16 * q) = aw;
    };

    v16f acc[RB];
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
        for (int r = 0; r < 16; ++r)
            acc[rb][r] = 0.f;

    v4u A[kRing], B[2][4];
    int cur = 0, next = kTile, after = 2 * kTile;                    // LDS offsets of this step's tile, the next one's, the one's after
    auto read_a = [&](int tile, int i) __attribute__((always_inline)) -> v4u {
        return *reinterpret_cast<const v4u *>(xrd + tile + 32 * (i % RB) * kPfRow + 16 * (i / RB));
    };

    WeightTables<S> tables;
    TablePieces<S <= 4 ? S : 2> pieces;                              // (unused, hence no registers, with more planes)
    WeightNibbles<S> nibbles;
    uint32_t pair[3][2], weights[8][2], sel, half, low[2], high[2];
    auto build = [&](auto U) __attribute__((always_inline)) {        // the table from c, piece by piece
        constexpr int u = decltype(U)::value;
        if constexpr (S <= 4) {
            if constexpr (u == 0)
                pieces.sums(c);
            else if constexpr (u == 1)
                pieces.round();
            else
                pieces.bytes(tables.t[0]);
        } else if constexpr (u == 0) {
            const uint32_t first[2] = {c[0], c[1] & 0xffffu};
            lut_build_tables<3>(first, tables.t[0]);
        } else if constexpr (u == 1) {
            const uint32_t second[2] = {(c[1] >> 16) | (c[2] << 16), c[2] >> 16};
            lut_build_tables<3>(second, tables.t[1]);
        } else if constexpr (S == 8) {
            const uint32_t third[1] = {c[3]};
            lut_build_tables<2>(third, tables.last);
        }
    };
    auto select = [&](auto P) __attribute__((always_inline)) {       // selector word p of w
        constexpr int p = decltype(P)::value;
        if constexpr (S <= 4) {
            if constexpr (p == 0)
                lut_nibble_pairs<S>(w, pair[0]);
            lut_nibble_word<S>(w, pair[0], nibbles.t[0], p);
        } else {
            const uint32_t first[3] = {w[0], w[1], w[2]}, second[3] = {w[3], w[4], w[5]};
            if constexpr (p == 0) {
                lut_nibble_pairs<3>(first, pair[0]);
                lut_nibble_pairs<3>(second, pair[1]);
            }
            lut_nibble_word<3>(first, pair[0], nibbles.t[0], p);
            lut_nibble_word<3>(second, pair[1], nibbles.t[1], p);
            if constexpr (S == 8) {
                const uint32_t third[2] = {w[6], w[7]};
                if constexpr (p == 0)
                    lut_nibble_pairs<2>(third, pair[2]);
                lut_nibble_word<2>(third, pair[2], nibbles.last, p);
            }
        }
    };
    auto look_up = [&](auto P, auto V, v4u (&Bn)[4]) __attribute__((always_inline)) {       // lut_look_up of p in pieces, and its place in the operand
        constexpr int p = decltype(P)::value, v = decltype(V)::value;
        uint32_t &w01 = weights[p][0], &w23 = weights[p][1];
        if constexpr (S == 4) {
            const LutTables<4> &t = tables.t[0];
            if constexpr (v == 0) {
                sel = (p < 4 ? nibbles.t[0].Q[p & 3] : nibbles.t[0].Q[p & 3] >> 4) & 0x07070707u;
                half = lut_halves(nibbles.t[0], p);
            } else if constexpr (v == 1) {
                low[0] = __builtin_amdgcn_perm(t.lo[1], t.lo[0], sel);
                high[0] = __builtin_amdgcn_perm(t.hi[1], t.hi[0], sel);
                low[1] = __builtin_amdgcn_perm(t.lo[3], t.lo[2], sel);
                high[1] = __builtin_amdgcn_perm(t.hi[3], t.hi[2], sel);
            } else {
                const uint32_t lo = __builtin_amdgcn_perm(low[1], low[0], half), hi = __builtin_amdgcn_perm(high[1], high[0], half);
                w01 = __builtin_amdgcn_perm(hi, lo, 0x05010400u);
                w23 = __builtin_amdgcn_perm(hi, lo, 0x07030602u);
            }
        } else {
            if constexpr (v == 0)
                lut_look_up<WeightTables<S>::H>(tables.t[0], nibbles.t[0], p, w01, w23);
            if constexpr (S > 4) {
                uint32_t e01, e23;
                if constexpr (v == 1)
                    lut_look_up<3>(tables.t[1], nibbles.t[1], p, e01, e23);
                else if constexpr (v == 2)
                    lut_look_up<2>(tables.last, nibbles.last, p, e01, e23);
                if constexpr (v > 0) {
                    w01 = __builtin_bit_cast(uint32_t, as_v2h(w01) + as_v2h(e01));
                    w23 = __builtin_bit_cast(uint32_t, as_v2h(w23) + as_v2h(e23));
                }
            }
        }
        if constexpr (v == Plan::kLook - 1) {
            Bn[p / 2][2 * (p & 1)] = w01;
            Bn[p / 2][2 * (p & 1) + 1] = w23;
        }
    };
    // Unit u of step ip.  kShare: odd steps are followed by a new pair of steps, whose table an even step has got ready (up to 4
    // planes, where it takes eight registers) but for the last piece; c is the line of the pair after the one being decoded.
    auto unit = [&](auto U, int ip, auto Odd, v4u (&Bn)[4]) __attribute__((always_inline)) {
        constexpr int u = decltype(U)::value;
        constexpr bool odd = decltype(Odd)::value;
        if constexpr (u < Plan::kNib) {
            store_x(next, u);
        } else if constexpr (u < Plan::kLoads) {
            if constexpr (u == Plan::kNib && kShare && odd && S <= 4)
                build(std::integral_constant<int, 2>{});
            select(std::integral_constant<int, u - Plan::kNib>{});
        } else if constexpr (u == Plan::kLoads) {
            next_words(ip + 1);
            load_words();
        } else if constexpr (u == Plan::kLoads + 1) {
            load_x();
        } else if constexpr (u < Plan::kCoeffs) {
            if constexpr (!kShare || (S > 4 ? odd : !odd && u < Plan::kTabs + 2))
                build(std::integral_constant<int, u - Plan::kTabs>{});
        } else if constexpr (u == Plan::kCoeffs) {
            if constexpr (!kShare || odd) {
                load_coefficients(line_of_next);
                line_of_next = load_line();
                next_line();
            }
        } else {
            look_up(std::integral_constant<int, (u - Plan::kLooks) / Plan::kLook>{}, std::integral_constant<int, (u - Plan::kLooks) % Plan::kLook>{}, Bn);
        }
    };
    // one step: its weights in Bc, the next one's decoded into Bn
    auto step = [&](int ip, auto Odd, const v4u (&Bc)[4], v4u (&Bn)[4]) __attribute__((always_inline)) {
        __builtin_amdgcn_sched_barrier(0);
        static_for<4 * RB>([&](auto I) __attribute__((always_inline)) {
            constexpr int i = decltype(I)::value, to = i + kAhead;
            acc[i % RB] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(v8h, A[i % kRing]), __builtin_bit_cast(v8h, Bc[i / RB]),
                                                                 acc[i % RB], 0, 0, 0);
            A[to % kRing] = to < 4 * RB ? read_a(cur, to) : read_a(next, to - 4 * RB);
            constexpr int first = Plan::kSlots.first[decltype(Odd)::value][i], units = Plan::kSlots.first[decltype(Odd)::value][i + 1] - first;
            static_for<units>([&](auto U) __attribute__((always_inline)) {
                unit(std::integral_constant<int, first + decltype(U)::value>{}, ip, Odd, Bn);
            });
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (i == 2 * RB - 1) {
                // (the LDS serves a wave in order: with no more than the kAhead youngest reads in flight, the tile is stored)
                asm volatile("s_waitcnt lgkmcnt(%0)\n\ts_barrier" ::"n"(kAhead) : "memory");
                __builtin_amdgcn_sched_barrier(0);
            }
        });
        const int t = cur;
        cur = next;
        next = after;
        after = t;
    };

    // -- prologue: the first step's activations stored and weights decoded, everything of the second in flight
    line_of_next = load_line();
    next_line();
    load_words();
    load_x();
    next_words(p0);
    load_coefficients(line_of_next);
    line_of_next = load_line();
    next_line();
    build_weight_tables<S>(c, tables);
    weight_nibbles<S>(w, nibbles);
#pragma unroll
    for (int q = 0; q < 4; ++q)
        B[0][q] = weight_operand<S>(tables, nibbles, q);
#pragma unroll
    for (int q = 0; q < NQ; ++q)
        store_x(cur, q);
    load_x();
    load_words();
    load_coefficients(line_of_next);
    line_of_next = load_line();
    next_line();
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kAhead; ++i)
        A[i] = read_a(cur, i);
    for (int ip = p0; ip < p_last; ip += 2) {
        step(ip, std::false_type{}, B[0], B[1]);
        step(ip + 1, std::true_type{}, B[1], B[0]);
    }
    if (!kShare && (p_last - p0) % 2 == 0)                           // an odd number of steps (the same for the whole workgroup)
        step(p_last, std::false_type{}, B[0], B[1]);

    // ---- D[i][jj] of a row block sits in lane jj + 32*((i/4)%2), register (i%4) + 4*(i/8)
    if (a.ksplit > 1) {
        float *mine = a.part + blockIdx.z * part_floats(M, N);
#pragma unroll
        for (int rb = 0; rb < RB; ++rb)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int m = m0 + 32 * rb + 8 * (r >> 2) + 4 * h + (r & 3);
                if (m < M && n < N)
                    mine[static_cast<size_t>(m) * N + n] = acc[rb][r];
            }
        return;
    }
    // through LDS, rows 528 bytes apart (lanes of both halves meet different banks), as many row blocks at a time as fit;
    // then thread t takes columns 8 (t % 32) .. + 7 of every sixteenth row
    constexpr int kOutRow = 2 * kPfBN + 16, kAtOnce = RB <= 6 ? RB : 4;
    static_assert(kAtOnce * 32 * kOutRow <= 3 * kTile, "the results of a turn in the activations' place");
    const int col = 8 * (tid & 31), cols = min(8, N - n0 - col);    // (none or fewer beyond the last column)
    uint16_t bias[8];
#pragma unroll
    for (int i = 0; i < 8; ++i)
        bias[i] = a.bias && i < cols ? a.bias[n0 + col + i] : 0;
    for (int turn = 0; turn < (RB + kAtOnce - 1) / kAtOnce; ++turn) {
        __syncthreads();                                             // (over the tiles, and the turn before)
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) {
            if (rb / kAtOnce != turn)                                // (uniform)
                continue;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int row = 32 * (rb % kAtOnce) + 8 * (r >> 2) + 4 * h + (r & 3);
                *reinterpret_cast<uint16_t *>(psm + row * kOutRow + 2 * (32 * wave + j)) = f2h(acc[rb][r]);
            }
        }
        __syncthreads();
        const int first = m0 + 32 * kAtOnce * turn, rows = min(min(32 * kAtOnce, m0 + 32 * RB - first), M - first);
        for (int row = tid >> 5; row < rows; row += 16) {
            v4u v = *reinterpret_cast<const v4u *>(psm + row * kOutRow + 2 * col);
            if (a.bias) {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    v[i] = static_cast<uint32_t>(hadd(static_cast<uint16_t>(v[i] & 0xffffu), bias[2 * i])) |
                           (static_cast<uint32_t>(hadd(static_cast<uint16_t>(v[i] >> 16), bias[2 * i + 1])) << 16);
            }
            uint16_t *const dst = a.out + static_cast<size_t>(first + row) * N + n0 + col;
            if (cols == 8) {
                *reinterpret_cast<v4u_any *>(dst) = v;               // (rows start anywhere: a global store wants no alignment)
            } else {
#pragma unroll
                for (int i = 0; i < 8; ++i)
                    if (i < cols)
                        dst[i] = static_cast<uint16_t>(i & 1 ? v[i / 2] >> 16 : v[i / 2] & 0xffffu);
            }
        }
    }
}

template <int S, int RB, bool kShare>
hipError_t launch_inst(const GemmArgs &a, hipStream_t st)
{
    constexpr int lds = 3 * 256 * kPfRow;
    {
        static std::mutex lock;
        static bool raised_on[16] = {};
        std::lock_guard<std::mutex> guard(lock);
        int dev = 0;
        if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 16)
            dev = 0;
        if (!raised_on[dev]) {
            const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(sbvr_gemm_lut_pipelined_kernel<S, RB, kShare>),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, lds);
            if (e != hipSuccess)
                return e;
            raised_on[dev] = true;
        }
    }
    const dim3 grid(static_cast<unsigned>((a.N + kPfBN - 1) / kPfBN), static_cast<unsigned>((a.M + 32 * RB - 1) / (32 * RB)),
                    static_cast<unsigned>(a.ksplit));
    hipLaunchKernelGGL((sbvr_gemm_lut_pipelined_kernel<S, RB, kShare>), grid, dim3(64 * kPfWaves), lds, st, a);
    return hipGetLastError();
}

template <int S, bool kShare>
hipError_t launch_rows(int rb, const GemmArgs &a, hipStream_t st)
{
    switch (rb) {
    case 5: return launch_inst<S, 5, kShare>(a, st);
    case 6: return launch_inst<S, 6, kShare>(a, st);
    case 7: return launch_inst<S, 7, kShare>(a, st);
    case 8: return launch_inst<S, 8, kShare>(a, st);
    default: return hipErrorInvalidConfiguration;
    }
}

template <int S>
hipError_t launch_planes(int rb, const GemmArgs &a, hipStream_t st)
{
    return a.steps_per_group % 2 == 0 ? launch_rows<S, true>(rb, a, st) : launch_rows<S, false>(rb, a, st);
}

}  // namespace

hipError_t launch_gemm_lut_pipelined(int S, int rb, const GemmArgs &a, hipStream_t st)
{
    switch (S) {
    case 2: return launch_planes<2>(rb, a, st);
    case 3: return launch_planes<3>(rb, a, st);
    case 4: return launch_planes<4>(rb, a, st);
    case 6: return launch_planes<6>(rb, a, st);
    case 8: return launch_planes<8>(rb, a, st);
    default: return hipErrorInvalidConfiguration;
    }
}
