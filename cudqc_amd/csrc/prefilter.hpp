// The raw cliques a maximal-set filter still has to look at (prefilter.hip).
#pragma once
#include <cstdint>
#include <vector>

#include "../../include/dqc.h"

namespace dqc {

// As dqc_fetch_batch_cliques (graph null: as dqc_fetch_cliques), without cliques that equal
// another one or lack exactly one vertex of another one: the maximal sets of what is left
// are those of all raw cliques. The order is not defined.
dqc_status fetch_candidates(dqc_handle* h, std::vector<int32_t>* graph, std::vector<int32_t>& sizes,
                            std::vector<int32_t>& ids);

}  // namespace dqc
