// The pair attention over pair columns, and where the pass is the faster form.
#include "pair_attn.h"

extern "C" int ga_pair_attention(const int32_t *type_pointer, int64_t n_types,
                                 const int64_t *by_type, const int64_t *dst_by_type,
                                 const int32_t *pair_pointer, const int32_t *nbr, const void *q,
                                 const void *k, const void *v, const void *att, const void *msg,
                                 void *m, float *lse, int64_t n_pairs, int64_t max_slots,
                                 int64_t heads, int64_t dim, int dtype, ga_stream_t stream) {
  if (!ga::pair_counts_ok(n_types, n_pairs, max_slots, heads, dim, dtype)) return GA_EINVAL;
  if (n_pairs == 0) return GA_OK;
  if (!type_pointer || !by_type || !dst_by_type || !pair_pointer) return GA_EINVAL;
  ga::PairArgs A{nullptr, nullptr, type_pointer, by_type, dst_by_type, pair_pointer, nbr, q, k, v,
                 att, msg, m, lse, (int)n_types};
  const int rc = ga::check_pairs(A, max_slots);
  if (rc != GA_OK) return rc;
  if (dtype == GA_F32)
    return ga::launch_pairs_dim<float, false>(A, n_pairs, heads * dim, dim, (hipStream_t)stream);
  return ga::launch_pairs_dim<ga::bf16_t, false>(A, n_pairs, heads * dim, dim, (hipStream_t)stream);
}

// Where the pass beats the three launches, from what the host knows.  A lane group walks
// rpg rows of a tile, four slots per dependent batch, and nobody helps it: the pass takes
// the longer of its share of the traffic and that chain, and large pairs come on top --
// taken as one and a half rows of the largest size on one group, between a lone large pair
// and many side by side.  The three launches pay for the pairs' rows in memory and for
// their own starts, but spread the slots evenly.  The figures (us; 0.72 per batch, 30 and
// 33 per 100 k pairs and 1 M edges of 256-byte rows) were fitted to the pass over pair columns.
// Over prepared tiles it is faster, one head of 64 fp32 features most (a group walks two
// rows, not four), so the line is on the launches' side: of 433 combinations of 500 to 1 M
// pairs of 2 to 256 slots in five layouts 39 take a form that is more than 5 % slower than the
// other, 37 of them the launches.  The operator as it runs, pass : launches, 1 x 64 fp32:
//   500 pairs of 16 / 32 / 64 / 256       23 : 34,   30 : 34,   45 : 36,  131 : 48
//   2,500 pairs of 32 / 64 / 256          35 : 44,   48 : 49,  131 : 73
//   10,000 pairs of 32 / 64 / 256         38 : 59,   52 : 73,  140 : 169
//   40,000 pairs of 64 / 256             141 : 181, 489 : 563
//   100,000 pairs of 3 on average, 0.3 % of 64 / 128 / 256    78 : 102,  87 : 103, 125 : 103
//   1 M pairs of 3, 0.3 % of 64 / 128 / 256                  392 : 653, 442 : 667, 585 : 690
extern "C" int ga_pair_attention_preferred(int64_t n_pairs, int64_t n_edges, int64_t max_slots,
                                           int64_t heads, int64_t dim, int dtype) {
  if (n_pairs <= 0 || n_edges < n_pairs || heads <= 0 || dim <= 0 || max_slots > 256) return 0;
  if (dtype != GA_F32 && dtype != GA_BF16) return 0;
  if ((heads * dim != 64 && heads * dim != 128) || (dim != 8 && dim != 16 && dim != 32 && dim != 64))
    return 0;
  const double rpg = (double)(heads * dim * (dtype == GA_F32 ? 4 : 2)) / 64;    // rows per lane group
  const double mean = (double)((n_edges / n_pairs + ga::kPairBatch - 1) / ga::kPairBatch);
  const double most = (double)((max_slots + ga::kPairBatch - 1) / ga::kPairBatch);
  const double p = 1e-3 * (double)n_pairs, e = 1e-3 * (double)n_edges, row = rpg / 4;
  const double share = (0.30 * p + 0.033 * e) * row, chain = 0.72 * rpg * mean;
  const double extra = most > mean ? 1.5 * 0.72 * (most - mean) : 0.0;
  const double pass = 20.0 + (share > chain ? share : chain) + extra;
  const double three = 36.0 + (0.43 * p + 0.033 * e) * row;
  return pass < three;
}
