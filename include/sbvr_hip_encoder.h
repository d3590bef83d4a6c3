/* Encoder search on the GPU (libsbvr_hip.so, gfx950).  Device pointers; the
 * launch goes to `stream` (a hipStream_t, NULL = default stream).  Return
 * values: 0 ok, -1 invalid argument, -2 unsupported shape, -3 launch error.
 */
#ifndef SBVR_HIP_ENCODER_H
#define SBVR_HIP_ENCODER_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/* mse[b, l] = mean over the G values of group b of min_p (data[b, g] - points[l, p])^2, for `groups`
 * groups and n candidate lines at once: data (groups, G) fp16, points (n, P) fp16 (the P = 2^S subset
 * sums of each line, 4-byte aligned), mse (groups, n) fp32.  Difference and square are rounded to fp16
 * and the minimum is taken there, as the reference's search does in its fp16 compute type
 * (sbvr/core.py:485-495, _data_diff_min_mse: `(data - candidate_matrix)**2`, `.min(dim=-1)`); the sum
 * over the group is fp32 in element order, divided by G (the reference: `.to(torch.float32).mean(dim=-1)`,
 * whose order of summation is torch's).  groups <= 65535, P a power of two up to 256 (S <= 8).
 * Replaces the error evaluation inside _search_coeff_bias_space (core.py:530-553), which
 * the reference runs for one group at a time (core.py:711-722). */
int sbvr_hip_encoder_group_mse_f16(const void *data, const void *points, float *mse, int groups, int G, int n, int P,
                                   void *stream);

/* The candidate lines of one group's search (sbvr/core.py:368-403) and their errors in one launch.  data: the group,
 * G fp16 values.  Lines 0 .. bs * ss * bases - 1: b[ib] + s[is] * base[ir, :] (fp16 product, fp16 sum), ir the fastest,
 * ib the slowest; behind them steps^S lines whose coefficient q is axes[q, i_q], the last axis fastest.  base
 * (bases, S), b (bs), s (ss), axes (S, steps): fp16.  lines (n, S) fp16 and mse (n) fp32 are written, mse as
 * sbvr_hip_encoder_group_mse_f16 writes it for the line's subset sums (fp32 sums rounded to fp16 once).  2 <= S <= 6, G
 * a multiple of 4 and at most 4096, at most 2^28 lines of either kind. */
int sbvr_hip_encoder_candidates_f16(const void *data, int G, const void *base, int bases, const void *b, int bs, const void *s,
                                    int ss, const void *axes, int steps, int S, void *lines, float *mse, void *stream);

/* The encoder's policy over `groups` groups in order (sbvr/core.py:555-653), on the device: rounds of two launches, each of
 * which takes the next group that the table does not serve through its search and settles what the groups behind it
 * see.  The caller brings, all on the device: data (groups, G) fp16; q95 and mean (groups) fp32, every group's 0.95
 * quantile and mean; table (table_lines, S) fp16; best (groups) fp32 and line (groups), the least error over the
 * table's lines and the first line that has it (infinity and -1 without lines); line_of (groups) and sel (groups, G), what
 * comes out; settled (groups), zeros; history, the errors of the searches so far, with room for one more per group; and
 * state, sbvr_hip_encoder_state_bytes() bytes: two slots of {int lines, misses, history, status, miss, unmet; uint64
 * found}.  Slot 0 starts as {lines in the table, groups so far that were no table hits, errors in `history`, 0, the first
 * group that misses, 0, all ones}.  Or with the last `unmet` groups to meet the table still, a window of them at a time as their turn
 * comes near: best and line are then over all lines for the groups in front of them (none of which need there be where the
 * table has lines), and miss is the first of those that misses, or groups - unmet.  A round reads slot (and
 * leaves it but for `found`) and writes the other.  Afterwards the slot that the last round wrote
 * holds the same; miss >= groups: nothing misses any more; status 1: group `miss` is left to the caller.
 * [0] and [1]: the plainer and the wider search: base (bases, S) and offsets fp16 as for
 * sbvr_hip_encoder_candidates_f16, axis_values values per axis of the grid.  scale_step, scale_narrow: 1 / number of scales,
 * 1 / what the wider search narrows their step by.  warmup, window, acceptable: lines before the table is used, errors in
 * the cut-off's mean, the least cut-off.  before: groups encoded before data's first.
 * lines: candidates of a search, for the launch's size (a search of more goes over its threads again).
 * 2 <= S <= 6, G a multiple of 4 and at most 4096, S * axis_values <= 4096. */
typedef struct {
    const void *data;
    const float *q95, *mean;
    void *table;
    float *best;
    int *line, *line_of, *sel;
    unsigned char *settled;
    void *state;
    double *history;
    const void *base[2], *offsets[2];
    int bases[2], n_offsets[2], axis_values[2];
    float scale_step, scale_narrow;
    int groups, G, warmup, window, table_lines;
    long long before;
    double acceptable;
} sbvr_hip_encoder_run;
size_t sbvr_hip_encoder_state_bytes(void);
/* The most scales a search of this space may have for the rounds to take it (a group with more is left to the caller), 0 where
 * they take no such search. */
int sbvr_hip_encoder_scales(int S, int G, int bases, int n_offsets, int axis_values);
int sbvr_hip_encoder_rounds_f16(const sbvr_hip_encoder_run *run, int S, int lines, int slot, int rounds, void *stream);

/* sel and line_of of groups first .. first + groups - 1 that are not settled, against the table line `line` names. */
int sbvr_hip_encoder_selectors_f16(const sbvr_hip_encoder_run *run, int S, int first, int groups, void *stream);

/* Activations to bit planes on the fly: x (M, K) fp16 -> bvr (K/32, M, S) uint32, bit k%32 of
 * bvr[k/32, m, j] = bit S-1-j of the selector of x[m, k] (point p of a line is the sum of the
 * coefficients j with bit S-1-j of p set, sbvr/core.py:345-351): the index of the first of the 2^S points of group
 * k/G (points (K/G, 2^S) fp16, the subset sums of that group's input coefficients) nearest to x[m, k],
 * difference and square in fp16 (the encoder's selector rule, sbvr/core.py:492-494).  The result, with
 * coeff_idx[g, m] = g and the input coefficients as coeff_cache, is the left operand of sbvr_hip_mm_T.
 * This is what the reference's _online_tranfrom / online_mm_T (sbvr/core.py:1021-1027, both return
 * None there) are placeholders for.  G a multiple of 32, K of G, S <= 8, M <= 65535. */
int sbvr_hip_online_encode_f16(const void *x, const void *points, uint32_t *bvr, int M, int K, int G, int S, void *stream);

/* The same encoding from the input coefficients themselves: lines (K/G, S) fp16, one line per group of K; the
 * subset sums are worked out in the launch (fp32 sum in the order of the coefficients, rounded to fp16 once).  Also
 * writes the line indices of the left operand, idx (K/G, M): idx[g, m] = g, uint8 (idx_bytes 1, K/G <= 256)
 * or uint16 (idx_bytes 2). */
int sbvr_hip_online_encode_lines_f16(const void *x, const void *lines, uint32_t *bvr, void *idx, int idx_bytes, int M, int K,
                                     int G, int S, void *stream);

/* Both in one: x (M, K) fp16 encoded against lines (K/G, Sl) as above, times the encoded weight (N, K) of r_bvr, r_idx and
 * r_cache (sbvr_hip_mm_T's right operand), plus bias (N) or NULL: out (M, N) fp16.  Where sbvr_hip_online_mm_T_scratch says 0 the
 * two calls by themselves are the way; elsewhere `scratch` is memory of the call's own of that many bytes, 16-byte aligned, that
 * nothing need clear. */
size_t sbvr_hip_online_mm_T_scratch(const uint32_t *r_bvr, const void *r_cache, int M, int N, int K, int Sl, int Sr, int G);
int sbvr_hip_online_mm_T(const void *x, const void *lines, const uint32_t *r_bvr, const void *r_idx, int r_idx_bytes, const void *r_cache,
                         const void *bias, void *out, int M, int N, int K, int Sl, int Sr, int G, int Lr, void *scratch,
                         size_t scratch_bytes, void *stream);

/* The dense weight of an encoded one (sbvr/core.py:926-949, decode()): out (N, k_out), out[n, k] = the sum of the
 * coefficients cache[idx[k / G, n], j] whose plane j is set at (n, k), added up in fp32, rounded to fp16 once and
 * converted to out_type (0 fp16, 1 bf16, 2 fp32).  bvr (K/32, N, S) uint32, idx (K/G, N) uint8 or uint16 (idx_bytes),
 * cache (L, S) fp16; k_out <= K leaves the padding of the last dimension out;
 * the elements of a group whose index is not below L are NaN.  A coefficient that is not finite counts as 0 * c = NaN
 * where its plane is not set, as in the product of the selector bits with the line.  Any S; G a multiple of 32, K of G. */
int sbvr_hip_decode_weight(const uint32_t *bvr, const void *idx, int idx_bytes, const void *cache, void *out, int out_type,
                           int N, int K, int k_out, int S, int G, int L, void *stream);

#ifdef __cplusplus
}
#endif

#endif
