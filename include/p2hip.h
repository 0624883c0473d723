/* libp2hip.so -- C ABI of the MI355X (gfx950) kernels for the ReBeL search hot path.
 *
 * Conventions shared by every entry point
 *   - plain pointers and sizes only; all pointers are DEVICE pointers unless named host_*;
 *   - H = 1326 hole-card combos, combo (a<b) at index a*(103-a)/2 + (b-a-1); float32
 *     data rows are H floats, row-major, contiguous; index arrays are int64; masks are
 *     one byte per element (0 / non-zero); float rows must be 8-byte aligned;
 *   - work is enqueued on `stream` (a hipStream_t, NULL = default stream); nothing
 *     synchronises, allocates or keeps a pointer after returning;
 *   - return value: 0 on success, otherwise a hipError_t (1 = invalid argument).
 *
 * The reference (phulin/poker2) has no FFI: the interface each function replaces is the
 * Python/Triton wrapper cited next to it (paths relative to the reference's src/p2/).
 */
#ifndef P2HIP_H
#define P2HIP_H

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

int p2hip_abi_version(void);
int p2hip_device_count(void);
const char* p2hip_error_string(int code);

/* ---- 7-card hand ranker -------------------------------------------------------- */

/* cards [n,7] ids 0..51 of elem_size bytes (1, 2 or 8) -> out[n] packed int32 score
 * (type nibble << 20 | five kicker nibbles).  Replaces rank_7_cards_single_batch_triton,
 * env/rules_triton.py:96-117 (kernel :617-632). */
int p2hip_rank7_cards(const void* cards, int elem_size, int64_t n, int32_t* out, void* stream);

/* cards [n,2,7] -> out[n] in {-1,0,1}, 1 = first hand stronger.  Replaces
 * compare_7_cards_single_batch_triton, env/rules_triton.py:78-93 (kernel :600-614). */
int p2hip_compare7_cards(const void* cards, int elem_size, int64_t n, int32_t* out, void* stream);

/* planes [n,4,13] bytes -> packed score.  flush_first = 1: flush suit is the first suit
 * with >= 5 ranks (env/rules_triton.py:229-242); 0: the fullest suit (env/rules.py:215-219).
 * Replaces create_comparison_vector + packing, env/rules.py:136-299, :406-407. */
int p2hip_rank7_planes(const uint8_t* planes, int64_t n, int32_t* out, int flush_first, void* stream);

/* planes [n,2,4,13] bytes -> out[n] in {-1,0,1}.  Replaces compare_7_single_batch
 * (env/rules.py:390-409) and compare_7_single_batch_triton (env/rules_triton.py:36-51). */
int p2hip_compare7_planes(const uint8_t* planes, int64_t n, int32_t* out, int flush_first, void* stream);

/* ---- river showdown --------------------------------------------------------------- */

/* Bytes of one per-board strength table (fixed). */
int64_t p2hip_showdown_table_bytes(void);

/* boards [m,5] ids of elem_size bytes (1,2,4,8).  Any of the three outputs may be NULL.
 *   mode 0: combos touching the board are ranked as 6-card hands; ranks_out [m,H] int32 =
 *           dense 1-based strength group ids            (rank_hands, env/rules.py:66-133)
 *   mode 1: 7 card ids, hole cards first, repeated ids count twice; ranks_out = packed scores
 *                                                 (rank_hands_triton, env/rules_triton.py:120-148)
 *   order_out [m,H] int64: stable ascending argsort of the scores;
 *   table_out [m, p2hip_showdown_table_bytes()]: what p2hip_showdown_both reads; replaces the
 *           HandRankData built by _init_hand_rank_data, search/cfr_evaluator.py:406-482. */
int p2hip_showdown_setup(const void* boards, int elem_size, int64_t m, int mode, int32_t* ranks_out,
                         int64_t* order_out, uint8_t* table_out, void* stream);

/* The same table from hands that are already in strength order, without a board: per row and
 * sorted position the hand's two cards c1_sorted, c2_sorted [m,H] int32 and its tie group
 * [L_idx, R_idx) [m,H] int32 -- the inputs of showdown_ev_triton, search/fused_cfr_triton.py:2271-2314.
 * bad [m] int32 receives 1 for a row that does not list each of the 1326 hands once with
 * 0 <= L <= k < R <= H (its table is filled with in-range values but means nothing), else 0. */
int p2hip_showdown_setup_sorted(const int32_t* c1_sorted, const int32_t* c2_sorted, const int32_t* L_idx,
                                const int32_t* R_idx, int64_t m, uint8_t* table_out, int32_t* bad, void* stream);

/* beliefs [m,2,H] -> out [m,2,H]: blocker-corrected showdown EV of both players per hand,
 * times potential[m,p] / scale[m].  table_row [m] (or NULL = identity) selects the board
 * table of each node.  Replaces _showdown_value_both / _showdown_value,
 * search/cfr_evaluator.py:484-601. */
int p2hip_showdown_both(const float* beliefs, const uint8_t* tables, const int64_t* table_row,
                        const float* potential, const float* scale, int64_t m, float* out, void* stream);

/* The same on rows of a node table: state k reads beliefs row node_rows[k] and writes out row node_rows[k], both
 * [rows,2,H] (NULL = identity); the rows are taken on trust. */
int p2hip_showdown_rows(const float* beliefs, const uint8_t* tables, const int64_t* table_row, const int64_t* node_rows,
                        const float* potential, const float* scale, int64_t m, float* out, void* stream);

/* ---- single-card chance node around the leaf network --------------------------------- */

/* For each of n public states (state i reads row root_indices[i] of pre_beliefs [*,2,H] and of
 * board [*,5] int64, -1 = empty slot; root_indices NULL = identity) and every card c not on its
 * board, in (i, c) ascending order: post_beliefs[s] = the ranges with the hands that hold c or
 * a board card removed, renormalised per player (uniform over the allowed hands when the sum
 * is <= 1e-12); board_samples[s] = the board with c in its first empty slot; root_lookup[s] = i.
 * sample_offsets [n+1] int64 (device) = prefix sums of 52 - cards on board.  source_rows = rows of
 * pre_beliefs / board, total_samples = rows the three outputs hold: a state whose row index lies
 * outside 0..source_rows-1 is skipped and no sample at or beyond total_samples is written, so
 * offsets that disagree with the boards cannot make the kernel leave its buffers; where a state
 * yields fewer samples than its share [sample_offsets[i], sample_offsets[i+1]) of the outputs (more
 * cards on its board than the offsets assume, no empty slot, a skipped row) the rest of the share is
 * filled with zeros and root_lookup with i, so no output row is left uninitialised.  Replaces the
 * expansion half of ChanceNodeHelper.single_card_chance_values,
 * search/chance_node_helper.py:394-443. */
int p2hip_chance_expand(const float* pre_beliefs, const int64_t* root_indices, const int64_t* board, int64_t n,
                        const int64_t* sample_offsets, int64_t source_rows, int64_t total_samples,
                        float* post_beliefs, int64_t* board_samples, int64_t* root_lookup, void* stream);

/* The same expansion written as rows of a value network's INPUT MATRIX: input_rows [total_samples, 2704]
 * in element type dtype (0 float32, 1 bfloat16, 2 float16), row s = the sample's 2 x 1326 ranges followed
 * by the 52-entry one-hot of its board (the state's cards and the dealt one) — what the reference builds
 * with a concatenation and a cast in front of its network (models/mlp/rebel_ffn.py forward; the ranges
 * are the `beliefs` of the MLPFeatures that search/chance_node_helper.py:445-456 assembles).
 * input_rows and pre_beliefs must be 16-byte aligned; board_samples may be NULL. */
int p2hip_chance_expand_input(const float* pre_beliefs, const int64_t* root_indices, const int64_t* board, int64_t n,
                              const int64_t* sample_offsets, int64_t source_rows, int64_t total_samples,
                              void* input_rows, int dtype, int64_t* board_samples, int64_t* root_lookup, void* stream);

/* A single-card chance node and the value network behind it in one call, in float32: expected [n,2,H] =
 * the mean over a state's samples (as p2hip_chance_expand makes them) of a network of `layers` linear
 * layers with ReLU between them whose input is a row of p2hip_chance_expand_input.  host_weights[l]
 * (device, [host_widths[l], columns] row-major, columns = 2704 for l = 0 and host_widths[l-1] after
 * it), host_biases[l] (device, or NULL for none), all 16-byte aligned; the last width is 2 H, the
 * others multiples of 32; 3 to P2HIP_NETWORK_MAX_LAYERS layers, at most P2HIP_NETWORK_MAX_SAMPLES samples.
 * `workspace`: 256-byte aligned, of p2hip_chance_network_workspace(...) bytes (-1: not a network this
 * call takes); its contents do not matter and mean nothing afterwards.  Everything that depends on the
 * weights is derived anew in every call.  Products are three of float16 halves under powers of two, a hidden unit's own
 * among them: errors as of float32 products for finite numbers, but an infinity may turn into NaN.  Every state needs a
 * sample (with total_samples = 0 nothing is written).  Replaces search/chance_node_helper.py:394-477 for such networks. */
#define P2HIP_NETWORK_MAX_LAYERS 16
#define P2HIP_NETWORK_MAX_SAMPLES ((1 << 23) - 1)
int64_t p2hip_chance_network_workspace(int64_t n, int64_t total_samples, const int32_t* host_widths, int layers);
int p2hip_chance_network(const float* pre_beliefs, const int64_t* root_indices, const int64_t* board, int64_t n,
                         const int64_t* sample_offsets, int64_t source_rows, int64_t total_samples,
                         const float* const* host_weights, const float* const* host_biases, const int32_t* host_widths,
                         int layers, void* workspace, int64_t workspace_bytes, float* expected, void* stream);

/* expected[i] = mean of hand_values [S,2,H] over samples sample_offsets[i] .. sample_offsets[i+1]
 * (index_add_ + divide of search/chance_node_helper.py:467-477). */
int p2hip_chance_mean(const float* hand_values, const int64_t* sample_offsets, int64_t n, float* expected,
                      void* stream);

/* Three-card (flop) chance node, flop_chance_values of search/chance_node_helper.py:219-357.
 * out [n, n_flops, 2, H]: the ranges of state i (row root_indices[i] of pre_beliefs [*,2,H], NULL =
 * identity) with the hands holding a card of flops[f] (int64 [n_flops,3]) removed, renormalised per
 * player (uniform over the 1176 surviving hands when the sum is <= 1e-12). */
int p2hip_flop_expand(const float* pre_beliefs, const int64_t* root_indices, int64_t n, const int64_t* flops,
                      int64_t n_flops, float* out, void* stream);

/* out [n,2,H] (+= if accumulate) sum_f weight[f] * mean_q hand_values[i][f][p][perms[q][h]]:
 * hand_values [n, n_flops, 2, H], perms int16 [n_perms <= 24, H] hand permutations, 4-byte aligned
 * (the suit-orbit mean of _avg_over_perms, :18-28, and the weighted flop sum, :352-357).  Evaluated as
 * mean_q Y[perms[q][h]] with Y = sum_f weight[f] * hand_values[i][f][p] summed in float64 - the same
 * number, since the permutations do not depend on the flop: a read stream and one permutation pass.
 * shares >= 1 splits the flops over that many workgroups per (state, player) - use it when
 * 2 * n alone leaves most of the GPU idle (a few hundred workgroups are enough); shares > 1 needs workspace [shares, n, 2, H] float32, whose
 * partial sums are added in ascending order (results do not depend on scheduling). */
int p2hip_perm_mean(const float* hand_values, int64_t n, int64_t n_flops, const int16_t* perms, int n_perms,
                    const float* weight, int accumulate, float* out, float* workspace, int shares, void* stream);

/* p2hip_perm_mean for the case of ALL 24 suit permutations (the rows of combo_suit_permutation_tensor,
 * env/card_utils.py:161-181): the mean over the orbit of a hand is the mean over its class of
 * starting hands (13 pairs, 78 suited, 78 offsuit), so
 * out[i][p][h] (+)= sum_f weight[f] * mean over the class of h of hand_values[i][f][p][.].
 * Same arguments otherwise; the class tables are built into the library. */
int p2hip_orbit_mean(const float* hand_values, int64_t n, int64_t n_flops, const float* weight, int accumulate,
                     float* out, float* workspace, int shares, void* stream);

/* p2hip_orbit_mean without the workspace argument.  No counterpart in the reference: it is for
 * callers that cannot allocate device memory (code under HIP graph capture, tight serving loops,
 * harnesses that forbid hipMalloc).  The partial sums of shares > 1 go to an array inside the
 * library (P2HIP_ORBIT_SCRATCH_FLOATS float32 = 16 MiB per GPU, held until the process ends); the
 * call allocates and frees nothing.  shares * n * 2 * 1326 floats must fit it: a larger request
 * returns 2 (hipErrorOutOfMemory) before anything is launched.  Same results, bit for bit, as
 * p2hip_orbit_mean with the same `shares`.  Every call on one GPU uses that GPU's array: calls
 * that overlap on one GPU (different streams, threads) race; calls on one stream do not.
 * The array's address on a device is resolved by the first call made with that device current
 * (hipGetSymbolAddress, which may load the code object): make that call OUTSIDE graph capture — a call
 * with n = 0 does the resolution and nothing else (null pointers allowed).  Later calls on the device
 * neither allocate nor resolve anything. */
#define P2HIP_ORBIT_SCRATCH_FLOATS (4 * 1024 * 1024)
int p2hip_orbit_mean_static(const float* hand_values, int64_t n, int64_t n_flops, const float* weight,
                            int accumulate, float* out, int shares, void* stream);

/* ---- either side of the search in data generation ------------------------------------------ */

/* Context features and board of RebelFeatureEncoder.encode (models/mlp/rebel_feature_encoder.py:55-127)
 * for m public states: context [m,4] float32 (16-byte aligned) = (to_act, (to_act - button) mod 2,
 * clamp(pot / max(starting_stack0 + starting_stack1, 1), 0, 10), committed chips differ and
 * actions_this_round > 0); board_out [m,5] = last_board where the state is encoded before its
 * chance event (pre_chance [m] bytes; NULL = pre_chance_all for every state), else board.
 * All inputs int64: [m] or [m,2] / [m,5]. */
int p2hip_encode_context(const int64_t* to_act, const int64_t* button, const int64_t* starting_stacks,
                         const int64_t* pot, const int64_t* committed, const int64_t* actions_this_round,
                         const uint8_t* pre_chance, int pre_chance_all, const int64_t* last_board,
                         const int64_t* board, int64_t m, float* context, int64_t* board_out, void* stream);

/* Chip amounts of the action bins, the first result of HUNLTensorEnv.legal_bins_amounts_and_mask
 * (env/hunl_tensor_env.py:348-405): amounts [m, n_bins + 3] = -1 for fold and call,
 * to_call + trunc(bin * pot) for each bet bin (legal or not), the actor's stack for all-in.
 * host_bins: at most 5 pot fractions in HOST memory. */
int p2hip_bet_amounts(const int64_t* to_act, const int64_t* stacks, const int64_t* committed, const int64_t* pot,
                      int64_t m, const float* host_bins, int n_bins, int64_t* amounts, void* stream);

/* The rows of the node table that go to the leaf network, and its answers coming back: the evaluator's
 * `beliefs[model_indices]` gather and `latest_values.index_copy_(0, model_indices, values)`
 * (search/cfr_evaluator.py:1030-1043, search/fused_sparse_cfr_evaluator.py:431-445), with the
 * conversion to and from the network's dtype folded in (under autocast the reference casts in separate
 * passes).  src / dst [total_rows, 2, 1326] float32; rows [k] int64 (entries outside [0, total_rows)
 * are skipped); dtype 0 = float32, 1 = bfloat16 (round to nearest even), 2 = float16.
 * gather : dst[i, 0:2652] = src[rows[i]] in dst_dtype; dst rows are dst_stride ELEMENTS apart, so the
 *          target may be the network's input matrix with further feature columns behind the ranges.
 * scatter: dst[rows[i]] = src[i, 0:2652] as float32; src rows are src_stride elements apart.
 * Both sides 8-byte aligned; strides even (float32) or a multiple of four (16-bit types). */
int p2hip_gather_leaf_rows(const float* src, const int64_t* rows, int64_t k, int64_t total_rows, void* dst, int dst_dtype,
                           int64_t dst_stride, void* stream);
int p2hip_scatter_leaf_rows(const void* src, int src_dtype, int64_t src_stride, const int64_t* rows, int64_t k, float* dst,
                            int64_t total_rows, void* stream);

/* Policy targets of CFREvaluator.training_data (search/cfr_evaluator.py:1392-1393; _pull_back,
 * search/sparse_cfr_evaluator.py:465-489): out [n_rows, H, num_actions] with
 * out[k,h,a] = policy_avg[c,h] for the child c of node rows[k] that action a leads to, 0 for
 * actions without a child.  policy_avg [total,H]; the three index arrays are [total] int64. */
int p2hip_policy_targets(const float* policy_avg, const int64_t* rows, int64_t n_rows, const int64_t* child_offsets,
                         const int64_t* child_count, const int64_t* action_from_parent, int num_actions, float* out,
                         void* stream);

/* ---- local best response -------------------------------------------------------------- */

/* One tree level of _best_response_values (search/cfr_evaluator.py:636-714), in place on
 * values [total,2,H]: for the parents parent_base .. parent_base+num_parents-1 that have
 * children (rows child_offsets[p] .. +child_count[p], at most max_children <= 8: a parent with more
 * is skipped), the player to act takes the
 * per-hand maximum over children where deviating_player[p] == to_act[p] and the policy-weighted
 * mean elsewhere; the other player gets the expectation of its child values under the
 * blocker-projected action probabilities.  Rows without children are left as they are (leaf
 * values).  Call once per level, deepest parents first.  All index arrays are [total] int64. */
int p2hip_best_response_level(float* values, const float* policy, const float* beliefs, const int64_t* to_act,
                              const int64_t* deviating_player, const int64_t* child_offsets,
                              const int64_t* child_count, int64_t parent_base, int64_t num_parents,
                              int max_children, void* stream);

/* ---- betting tree on the device ----------------------------------------------------------- */

/* A node is a row of p2hip_tree_node_columns() int64 (21): street, to_act, button, pot, stack0,
 * stack1, committed0, committed1, min_raise, actions_this_round, is_allin0, is_allin1,
 * starting_stack0, starting_stack1, done, raises, scale (float32 bits), root row, parent row (-1),
 * action from parent (-1), fold reward (float32 bits).  Two launches per level replace the host
 * depth loop over HUNLTensorEnv (search/sparse_cfr_evaluator.py:142-306; rules of
 * env/hunl_tensor_env.py:348-423, 684-724, 766-992); the caller prefix-sums count_out in
 * between.  host_bins: bet fractions of the pot, at most 5, in HOST memory. */
int64_t p2hip_tree_node_columns(void);

/* legal_out [n, n_bins+3] bytes: legal action bins (fold, call, bets..., all-in) of every node;
 * count_out [n]: children the node gets (0 unless `expand`; 0 below the root level when the
 * node's betting round has just closed).  max_raises < 0: no cap on bets and raises per round. */
int p2hip_tree_legal(const int64_t* nodes, int64_t n, const float* host_bins, int n_bins, int max_raises,
                     int is_root_level, int expand, uint8_t* legal_out, int64_t* count_out, void* stream);

/* Children of the n parents (global rows parent_row_base ..), action ascending, written from row
 * child_start[i] of `children` on (exclusive prefix sums of count_out). */
int p2hip_tree_step(const int64_t* parents, int64_t n, int64_t parent_row_base, const float* host_bins, int n_bins,
                    int max_raises, int64_t bb, int is_root_level, const int64_t* child_start, int64_t* children,
                    void* stream);

/* ---- unblocked (card-compatible) mass --------------------------------------------- */

/* target [rows,H] -> out [rows,H] = max(S - cs[a] - cs[b] + t, 0).  Replaces
 * calculate_unblocked_mass (env/card_utils.py:196-222) and unblocked_mass_triton
 * (search/fused_cfr_triton.py:1110-1157). */
int p2hip_unblocked_mass(const float* target, int64_t rows, float* out, void* stream);

/* beliefs [total,2,H], to_act [total]; out[r] = unblocked(beliefs[r, to_act[r] ^ opponent])
 * for r < top.  Replaces unblocked_mass_opp_at_parents_triton,
 * search/fused_cfr_triton.py:1067-1107. */
int p2hip_unblocked_mass_by_player(const float* beliefs, const int64_t* to_act, int64_t top, int opponent,
                                   float* out, void* stream);

/* out[c] = d > eps ? unblocked(numer[c]) / d : 0, d = unblocked(denom[parent_index[c]])
 * (parent_index NULL = identity).  Replaces unblocked_mass_ratio_indirect_triton /
 * unblocked_mass_ratio_triton, search/fused_cfr_triton.py:1499-1602. */
int p2hip_unblocked_mass_ratio(const float* numer, const float* denom, const int64_t* parent_index,
                               int64_t rows, float eps, float* out, void* stream);

/* The same quotient from denominators that are already unblocked masses: d = denom_unblocked[parent_index[c]]
 * ([parents,H], e.g. from p2hip_unblocked_mass).  Siblings share their parent's row, so its card sums are
 * taken once per parent; the reference passes precomputed denominator statistics for the same purpose
 * (denom_stats of unblocked_mass_ratio_indirect_triton, search/fused_cfr_triton.py:1499-1556). */
int p2hip_unblocked_mass_ratio_of(const float* numer, const float* denom_unblocked, const int64_t* parent_index,
                                  int64_t rows, float eps, float* out, void* stream);

/* ---- per-operation CFR kernels (search/fused_cfr_triton.py) ------------------------- */
/* Scalars that depend on the iteration number are 0-D device tensors (const float*). */

/* fused_dcfr_update_with_tensors_ :200-235 (kernel :71-120).  n = element count (even).
 * positive_out may be NULL. */
int p2hip_dcfr_update(float* cumulative_regrets, float* regret_weight_sums, const float* regrets,
                      const float* t_alpha_num, const float* t_beta_num, const float* t_alpha_den,
                      const float* t_beta_den, int64_t n, int apply_dcfr, int cfr_plus, float* positive_out,
                      void* stream);

/* fused_block_and_normalize_beliefs_ :286-335.  target has rows*1 rows of H; row r uses
 * mask / fallback row r / players_per_row. */
int p2hip_block_and_normalize(float* target, const uint8_t* allowed, const float* allowed_prob, int64_t rows,
                              int players_per_row, float eps, void* stream);

/* fused_regret_matching_divide_ :369-399 */
int p2hip_regret_matching_divide(const float* positive, const float* denom, const float* fallback, float* out,
                                 int64_t n, float eps, void* stream);

/* fused_weight_child_values :438-477; values/out [m,2,H] */
int p2hip_weight_child_values(const float* values, const int64_t* prev_actor, const float* policy_hero,
                              const float* policy_opp, float* out, int64_t m, void* stream);

/* fused_update_average_values_with_tensors_ :538-560 */
int p2hip_update_average_values(float* values_avg, const float* latest, const float* old_w, const float* new_w,
                                const float* inv_total, int64_t n, void* stream);

/* fused_avg_values_zero_sum_ :623-668; ignore_mask [nodes] bytes or NULL */
int p2hip_avg_values_zero_sum(float* values_avg, const float* latest, const float* beliefs,
                              const uint8_t* ignore_mask, const float* old_w, const float* new_w,
                              const float* inv_total, int64_t nodes, int enforce_zero_sum, void* stream);

/* fused_regret_tail_ :712-766; writes rows [bottom,total) of regrets */
int p2hip_regret_tail(float* regrets, const float* values_achieved, const float* actor_values,
                      const float* src_weights, const int64_t* parent_index, const int64_t* prev_actor,
                      int64_t bottom, int64_t total, void* stream);

/* fused_average_policy_mix_with_tensors_ :879-914 */
int p2hip_average_policy_mix(float* policy_probs_avg, const float* policy_probs, const float* self_reach,
                             const float* self_reach_avg, const int64_t* to_act, const int64_t* parent_index,
                             const float* old_w, const float* new_w, const float* total_w, int64_t bottom,
                             int64_t total, float eps, void* stream);

/* fused_parent_sum :1279-1313 -> out [num_parents,H] */
int p2hip_parent_sum(const float* values, const int64_t* child_offsets, const int64_t* child_count,
                     int64_t num_parents, float* out, void* stream);

/* fused_sibling_sum :1355-1398 -> out [num_children,H], row = child - bottom */
int p2hip_sibling_sum(const float* values, const int64_t* child_offsets, const int64_t* child_count,
                      int64_t num_parents, int64_t bottom, float* out, void* stream);

/* fused_divide_by_parent_sum_ :1316-1352; out may alias pos or fallback */
int p2hip_divide_by_parent_sum(const float* pos, const float* fallback, const float* parent_sum,
                               const int64_t* parent_index, float* out, int64_t num_children, float eps,
                               void* stream);

/* fused_model_values_mix_with_tensors :1658-1680 */
int p2hip_model_values_mix(const float* hand_values, const float* last_values, const float* onon,
                           const float* oon, float* out, int64_t n, void* stream);

/* fused_model_values_mix_zero_sum :1739-1775; tensors [rows,2,H] */
int p2hip_model_values_mix_zero_sum(const float* hand_values, const float* last_values, const float* beliefs,
                                    const float* onon, const float* oon, float* out, int64_t rows,
                                    int enforce_zero_sum, void* stream);

/* fused_weighted_parent_sum :1838-1889; child_offsets/count already sliced to the depth */
int p2hip_weighted_parent_sum(float* values, const int64_t* prev_actor, const float* policy_hero,
                              const float* policy_opp, const int64_t* child_offsets, const int64_t* child_count,
                              int64_t num_parents, int64_t parent_base, void* stream);

/* fused_reach_weights_depth_ :1944-1986; rows [start,end) */
int p2hip_reach_weights_depth(float* reach, const float* policy, const uint8_t* allowed_mask,
                              const int64_t* parent_index, const int64_t* prev_actor, int64_t start, int64_t end,
                              void* stream);

/* fused_deep_beliefs_ :2039-2092; rows [n_roots,total) are written */
int p2hip_deep_beliefs(float* out, const float* root_beliefs, const float* reach, const float* allowed_prob,
                       const int64_t* root_index, int64_t n_roots, int64_t total, float eps, void* stream);

/* policy_probs_sample <- where(t_sample == *t_now, policy_probs, policy_probs_sample),
 * search/fused_sparse_cfr_evaluator.py:494-499 */
int p2hip_sample_snapshot(const float* policy_probs, float* policy_probs_sample, const int64_t* t_sample,
                          const int64_t* t_now, int64_t total, void* stream);

/* ---- a family, or a level of the tree, per launch ------------------------------------ */

/* What the methods of search/fused_sparse_cfr_evaluator.py compose of the operations above, in the same roundings, for
 * a whole tree: children of a parent p are rows child_offsets[p] .. + child_count[p] - 1, at most max_children <= 8 (a
 * parent that has more children than claimed may be left alone). */

/* compute_instantaneous_regrets (:312-349): achieved, expected, beliefs [T,2,H] -> regrets [T,H]; parents < top, rows <
 * bottom zero */
int p2hip_family_regrets(const float* achieved, const float* expected, const float* beliefs, const int64_t* to_act,
                         const int64_t* prev_actor, const int64_t* child_offsets, const int64_t* child_count,
                         int64_t bottom, int64_t top, float* regrets, void* stream);

/* the same, added to the cumulative regrets as p2hip_dcfr_update does instead of stored */
int p2hip_family_regret_update(const float* achieved, const float* expected, const float* beliefs, const int64_t* to_act,
                               const int64_t* prev_actor, const int64_t* child_offsets, const int64_t* child_count,
                               int64_t bottom, int64_t top, float* cumulative, float* weights, const float* t_alpha_num,
                               const float* t_beta_num, const float* t_alpha_den, const float* t_beta_den, int apply_dcfr,
                               int cfr_plus, void* stream);

/* the regret matching of update_policy (:201-218): policy[c] = max(cumulative[c], 0) / family sum, fallback[c] where
 * that is <= eps */
int p2hip_family_regret_matching(const float* cumulative, const float* fallback, const int64_t* child_offsets,
                                 const int64_t* child_count, int64_t top, int max_children, float eps, float* policy,
                                 void* stream);

/* update_average_policy (:355-398): the mix, then its division by the family sum; weights as device scalars */
int p2hip_family_average_policy(const float* policy, float* policy_avg, const float* reach, const float* reach_avg,
                                const int64_t* to_act, const int64_t* child_offsets, const int64_t* child_count,
                                const float* old_w, const float* new_w, const float* total_w, int64_t bottom, int64_t top,
                                int max_children, float eps, void* stream);

/* reach weights and ranges of every row below the n_roots roots (_calculate_reach_weights and _propagate_all_beliefs of a
 * whole tree of at most 64 levels); the nodes of a root share their allowed hands */
#define P2HIP_TREE_MAX_DEPTH 64
int p2hip_tree_reach_beliefs(float* reach, const float* policy, const uint8_t* allowed, const float* allowed_prob,
                             const int64_t* parent_index, const int64_t* prev_actor, const int64_t* root_index,
                             float* beliefs, int64_t n_roots, int64_t total, int depth, float eps, void* stream);

/* compute_expected_values (:242-306) of parents base .. base + n - 1, all of one level, from the level below */
int p2hip_level_expected_values(float* values, const float* policy, const float* beliefs, const int64_t* to_act,
                                const int64_t* child_offsets, const int64_t* child_count, int64_t base, int64_t n,
                                int max_children, float eps, void* stream);

/* ---- before the first iteration and after the last ------------------------------------ */

/* constant rows of a new state of `total` nodes, the first n_roots of them roots: uniform [T,H] = 1 / children of the
 * parent (0 for roots); reach, reach_avg [T,2,H] = 1 for roots, else 0; latest, values_avg [T,2,H] = reward, -reward of
 * the two players at folds, else 0 (search/sparse_cfr_evaluator.py:240-306) */
int p2hip_subgame_rows(const int64_t* parent_index, const int64_t* child_count, const uint8_t* fold_mask,
                       const float* reward, int64_t n_roots, int64_t total, float* uniform, float* reach, float* reach_avg,
                       float* latest, float* values_avg, void* stream);

/* board [roots,5] (-1 = not dealt): allowed [T,H] = no card of the hand on the board of row r's root, prob [T,H] uniform
 * over these hands (search/cfr_evaluator.py:780-815) */
int p2hip_allowed_hands(const int64_t* board, const int64_t* root_index, int64_t total, uint8_t* allowed, float* prob,
                        void* stream);

/* initialize_policy_and_beliefs (search/cfr_evaluator.py:830-886) for a uniform policy over the legal actions
 * (legal_mask [T,actions]) of a tree of `depth` <= P2HIP_TREE_MAX_DEPTH levels: roots [n_roots,2,H] = the roots' ranges
 * (not the rows of `beliefs`), root rows of `reach` read, everything else of the six tensors written */
int p2hip_uniform_start(const float* roots, const uint8_t* allowed, const float* allowed_prob, const int64_t* parent_index,
                        const int64_t* prev_actor, const int64_t* root_index, const uint8_t* legal_mask, int actions,
                        int64_t n_roots, int64_t total, int depth, float eps, float* policy, float* policy_avg,
                        float* reach, float* reach_avg, float* beliefs, float* beliefs_avg, void* stream);

/* out [T,2,H] = values at leaves (clamped to [-1,1] if `clamp`), 0 elsewhere */
int p2hip_leaf_rows(const float* values, const uint8_t* leaf_mask, int64_t total, int clamp, float* out, void* stream);

/* *found = 1 if one of n (even) floats is infinite or NaN, else untouched */
int p2hip_any_nonfinite(const float* x, int64_t n, int32_t* found, void* stream);

/* ---- one kernel = one CFR iteration ------------------------------------------------- */

/* Device pointers of one subgame batch.  Tree arrays and state tensors are the evaluator's
 * own (row-major over all nodes of all roots); the rest is derived once per subgame:
 *   node_flags [total] bytes: bit0 = river showdown row, bit1 = terminal row, bit2 = the row has children,
 *             bit3 = childless row whose ranges feed a leaf evaluation (a showdown row, or a row the caller's
 *             leaf network is asked about); bits 2 and 3 are read by lean launches only; bit4 = latest and values_avg of the row are one number per
 *             player, whatever the hand (a fold leaf; read by p2hip_cfr_iteration_shared only)
 *   root_parent_offsets [roots+1], root_parents: rows that have children, per root, ascending
 *   root_showdown_offsets [roots+1], root_showdown_nodes: river showdown rows per root
 *   tables [roots, p2hip_showdown_table_bytes()] (NULL when no row is a showdown)
 *   potential [total,2] float, scale [total] float: showdown pay-off factors per row
 *   scratch [total,H] float workspace (may be NULL when reach_avg_prev is given)
 *   fscal[8]: t^alpha, t^beta, t^alpha+1, t^beta+1, mix_old, mix_new, mix_old+mix_new, 1/(mix_old+mix_new)
 *   iscal[8]: t, apply_dcfr, cfr_plus, average_policy_is_copied, enforce_zero_sum, update_average_values,
 *             cfr_avg (regret weights and showdown values from beliefs_avg), linear (regrets of player t mod 2
 *             dropped, no discount) */
typedef struct P2HipIterArgs {
  const int64_t* child_offsets;
  const int64_t* child_count;
  const int64_t* to_act;
  const uint8_t* node_flags;
  const int64_t* root_parent_offsets;
  const int64_t* root_parents;
  const int64_t* root_showdown_offsets;
  const int64_t* root_showdown_nodes;
  const int64_t* t_sample;
  const uint8_t* allowed;
  const float* allowed_prob;
  const uint8_t* tables;
  const float* potential;
  const float* scale;
  float* policy;
  float* policy_avg;
  float* policy_sample;
  float* cum;
  float* wsum;
  float* beliefs;
  float* beliefs_avg;
  float* reach;
  float* reach_avg;
  float* latest;
  float* values_avg;
  float* scratch;
  const float* fscal;
  const int64_t* iscal;
  /* Optional work items (both NULL: one item per root, item w = root w, n_items = roots).
   * root_parent_offsets / root_showdown_offsets then have n_items + 1 entries and delimit, per item,
   * the families and showdown rows one workgroup walks; item_root [n_items] names the root an item
   * belongs to.  With few roots a root's tree may be cut at a level into a top item (item_top = 1: the
   * families and showdown rows above the cut) and one subtree item per node of the cut level that has
   * children (item_top = 0); every family and showdown row belongs to exactly one item.  An iteration
   * is then four launches: all items with phases 4, top items with 8, subtree items with 8|2, top items
   * with 2 (the regret part of a family reads rows that the reach / belief part of the family above
   * rewrites, so it runs everywhere first).  The tops may be cut again the same way (tiers of items:
   * reach / belief parts tier by tier downwards, value parts upwards; two launches more per cut). */
  const int64_t* item_root;
  const uint8_t* item_top;
  /* Optional, [total,2,H]: reach_avg as the PREVIOUS iteration left it, in a buffer of its own.  The
   * average-policy mix (search/fused_sparse_cfr_evaluator.py:355-398) weighs the old average policy by the
   * parent's reach_avg from before this iteration; with NULL the kernel saves that row in `scratch`
   * before it overwrites reach_avg in place.  A caller that keeps two reach_avg buffers and swaps them
   * from iteration to iteration passes the other one here and saves a row write and a row read per
   * parent.  Root rows of both buffers hold the roots' reach (1); must differ from reach_avg. */
  const float* reach_avg_prev;
} P2HipIterArgs;

/* One workgroup per root runs the whole iteration of FusedSparseCFREvaluator.cfr_iteration
 * (search/fused_sparse_cfr_evaluator.py:478-533; base search/cfr_evaluator.py:1330-1381) with
 * cfr_avg = False: sample snapshot, instantaneous regrets, DCFR update, regret matching, reach,
 * beliefs, average policy, reach_avg, beliefs_avg (phases bit 0; bit 2 = the regret part alone, bit 3 = the
 * reach / belief / average-policy part alone); showdown leaf values, value backup, average values
 * (phases bit 1).  phases bit 4 (16) marks a LEAN iteration, for callers that run many iterations and
 * look at the state only after the last (evaluate_cfr, search/cfr_evaluator.py:1497-1528): the reach /
 * belief part then stores only rows that a later part of this iteration or the next iteration reads —
 * reach and reach_avg of rows with children, beliefs of rows with children or a leaf evaluation
 * (node_flags bits 2, 3), beliefs_avg only under cfr_avg or enforce_zero_sum.  The rows left out are
 * functions of rows that are kept: one iteration without the bit afterwards leaves all eleven tensors
 * bit-identical to a run that never set it.  host_args is a HOST pointer to a struct of device
 * pointers; n_items = workgroups to launch (= roots unless the work-item lists are given);
 * max_children = largest child count in the tree (<= 8). */
int p2hip_cfr_iteration(const P2HipIterArgs* host_args, int64_t n_items, int max_children, int phases,
                        void* stream);

/* p2hip_cfr_iteration that moves fewer bytes where rows of the state repeat one another.
 *
 * range_rows (optional, [total], from p2hip_range_rows): reach, reach_avg, beliefs and beliefs_avg of the player
 *   who did not act on the way into a row are the numbers of an earlier row, bit for bit, back to that player's
 *   last action (or to the row right under the root).  range_rows[c] names it in the [total*2] row space.  With it
 *   every iteration reads those rows there and a lean iteration (bit 4) stores them only there; leaves a network
 *   is asked about (node_flags 8 without 1) and beliefs_avg under enforce_zero_sum keep both rows.
 * phases bit 5 (32): rows flagged 16 in node_flags (fold leaves: one number per player in latest and values_avg,
 *   whatever the hand) are read through their first two entries; a lean iteration stores only those two of
 *   values_avg.  After lean iterations with the bit, one iteration with the bit and without bit 4 makes every
 *   row whole again.
 * leaf_prev (optional, [total,2,H]): beliefs (beliefs_avg under cfr_avg) as the previous iteration left them, where
 *   that was another buffer than the one in host_args.
 * phases bit 6 (64): one walk per family instead of three (bit 7, 128, with it exactly if iscal[6] is set): regrets,
 *   policy, ranges, the value of the showdown child, and the backup of families whose children are all leaves, with
 *   phases bit 0; the backup of the others with bit 1.  Needs bits 4 and 5, range_rows, reach_avg_prev, at most five
 *   children per parent, at most one showdown child among siblings (not checked here: it is a property of the
 *   tree), no enforce_zero_sum, and two range buffers: leaf_prev is read and leaf_next written in place of
 *   beliefs (beliefs_avg under cfr_avg) of host_args; both hold the roots' ranges (the walk copies them on).
 *   Bits 2 and 3 do not apply: tiers of work items take bit 0 downwards and bit 1 upwards.
 * phases bit 8 (256): a lean iteration stores the rows that range_rows and bit 5 spare all the same, for a caller
 *   whose own code (a leaf network with the node table in hand) reads the state between the parts of an iteration;
 *   reads are as without it.  Not with bit 6.
 * The state after a closing iteration without bits 4 and 6 is bit-identical to p2hip_cfr_iteration's. */
int p2hip_cfr_iteration_shared(const P2HipIterArgs* host_args, const int32_t* range_rows, const float* leaf_prev,
                               float* leaf_next, int64_t n_items, int max_children, int phases, void* stream);

/* range_rows of a tree: parent_index [total] (rows numbered top-down, the n_roots roots first), to_act [total]. */
int p2hip_range_rows(const int64_t* parent_index, const int64_t* to_act, int64_t n_roots, int64_t total, int32_t* out,
                     void* stream);

/* Copy 8 floats and 8 int64 from HOST arrays into the device arrays fscal[8] / iscal[8] read by
 * p2hip_cfr_iteration.  The values travel as kernel arguments: the host arrays may be reused as
 * soon as the call returns.  Plays the role of TScalars.update, search/fused_cfr_triton.py:2131-2158. */
int p2hip_write_scalars(float* fscal, int64_t* iscal, const float* host_f, const int64_t* host_i, void* stream);

/* dst[0..n) (device, n <= 8) = host_values[0..n): the values travel as kernel arguments, in
 * stream order, so the scalar-taking wrappers (fused_dcfr_update_ etc., fused_cfr_triton.py:123-197)
 * need no host-to-device copies.  No counterpart in the reference, which passes Python floats to
 * Triton. */
int p2hip_upload_floats(float* dst, const float* host_values, int n, void* stream);

/* ---- measurement aid ------------------------------------------------------------------------ */

/* No counterpart in the reference and not on the search path: a structure-free element-wise stream over
 * n_read input and n_write output arrays of `pairs` float2 each (array k starts k * pairs float2 after the
 * base pointer), for (n_read, n_write) in {(5,7), (1,1), (2,0), (0,2)}; non_temporal != 0 marks every access
 * non-temporal.  bench.py times it to report what HBM gives a kernel of the iteration kernel's read / write
 * mix on the same machine. */
int p2hip_stream_probe(const float* in, float* out, int64_t pairs, int n_read, int n_write, int non_temporal,
                       void* stream);

/* ---- placement aid --------------------------------------------------------------------------- */

/* No counterpart in the reference (PyTorch's allocator places its tensors).  The iteration kernel writes
 * about ten tensors at once, and the card's memory takes that 10 % faster when the written tensors lie in
 * two different thirds (~96 GiB each) of its physical address space instead of one.  Where an allocation
 * lies physically is not visible, but it can be measured and steered:
 *
 * p2hip_placement_probe: time of one launch (ms, mean of `reps`, 1..64) of a row-streaming kernel - 12 rows
 *   of 1326 floats read and 8 written per node - whose 20 arrays are dealt alternately to the buffers `a`
 *   and `b` (ten arrays spread over the first `bytes_each` bytes of each; at least 14 MB each; contents
 *   are OVERWRITTEN).  Two buffers in different thirds take about a fifth less than two halves of one
 *   buffer, which is the comparison to make.  Synchronises the stream.
 * p2hip_device_reserve / _release: `bytes` of device memory from hipMalloc, untouched, to be HELD while
 *   something else is allocated so that it lands elsewhere; out of memory: the HIP error code, *out =
 *   NULL, nothing left pending.  Release synchronises the device. */
int p2hip_placement_probe(void* a, void* b, int64_t bytes_each, int reps, float* ms_out, void* stream);
int p2hip_device_reserve(int64_t bytes, void** out);
int p2hip_device_release(void* block);

#ifdef __cplusplus
}
#endif
#endif /* P2HIP_H */
