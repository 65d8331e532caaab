// The packing pass (spx::pack_place) on the host, thread by thread, after a service pass that counts and ranks the
// running slots as the kernels do.
#include <algorithm>
#include <cstring>
#include <vector>

#include "../../spectrum_amd/csrc/spx_kernels.h"

using namespace spx;

// `launches` packed launches over one pool: state[l * span + s] is the query of slot s (whole waves of one query, -1:
// idle) and run[l * span + s] whether it runs.  The waves are counted in the order given.  Returns 0, or which check of
// launch l failed: a running slot missing from its query's part, a place beyond the parts that is not -1, or a write
// outside the list.
extern "C" int pack_check(int launches, long span, long list_span, int n_queries, const int* queue, int n_queue, const int* state, const int* run,
                          const int* wave_order, int* failed_launch)
{
   const size_t guard = 4096;
   std::vector<int32_t> active((size_t)span), slot_q((size_t)span), rank((size_t)span), list((size_t)list_span + guard);
   std::vector<uint32_t> n_running(2 * (size_t)n_queries);
   Launch L;
   std::memset((void*)&L, 0, sizeof(L));
   L.queue = queue;
   L.n_queue = n_queue;
   L.n_queries = n_queries;
   L.active = active.data();
   L.slot_q = slot_q.data();
   L.rank = rank.data();
   L.n_running = n_running.data();
   L.list = list.data();
   int packed = 0;
   for (int l = 0; l < launches; l++, packed = 1 - packed) {
      *failed_launch = l;
      std::fill(list.begin(), list.end(), -7);
      for (long s = 0; s < span; s++) {
         active[s] = run[l * span + s] ? SLOT_RUN : SLOT_IDLE;
         slot_q[s] = state[l * span + s];
      }
      for (long w = 0; w < span / 64; w++) {   // service_slot's last part
         const long s0 = 64L * wave_order[w];
         uint32_t n = 0;
         for (int k = 0; k < 64; k++) n += active[s0 + k] == SLOT_RUN;
         if (n == 0) continue;
         uint32_t& count = n_running[(size_t)packed * n_queries + slot_q[s0]];
         uint32_t base = count;
         count += n;
         for (int k = 0; k < 64; k++)
            if (active[s0 + k] == SLOT_RUN) rank[s0 + k] = (int32_t)base++;
      }
      for (long s = 0; s < span; s++)   // before the pass writes: every place it is about to write lies in the list
         if (active[s] == SLOT_RUN) {
            uint64_t start = 0;
            for (int k = 0; k < n_queue && queue[k] != slot_q[s]; k++) start += (n_running[(size_t)packed * n_queries + queue[k]] + 63u) & ~63u;
            if (start + (uint64_t)rank[s] >= (uint64_t)list_span) return 3;
         }
      const uint64_t n_threads = (uint64_t)(std::max(span, list_span) + 255) / 256 * 256;
      for (uint64_t i = 0; i < n_threads; i++) pack_place(&L, packed, (uint64_t)span, (uint64_t)list_span, i, n_threads);
      size_t place = 0;
      for (int k = 0; k < n_queue; k++) {
         std::vector<int32_t> want, got;
         for (long s = 0; s < span; s++)
            if (active[s] == SLOT_RUN && slot_q[s] == queue[k]) want.push_back((int32_t)s);
         for (size_t i = 0; i < want.size(); i++) got.push_back(list[place + i]);
         std::sort(got.begin(), got.end());
         if (got != want) return 1;
         for (place += want.size(); place % 64 != 0; place++)
            if (list[place] != -1) return 2;
      }
      for (; place < (size_t)list_span; place++)
         if (list[place] != -1) return 2;
      for (size_t i = 0; i < guard; i++)
         if (list[(size_t)list_span + i] != -7) return 3;
   }
   return 0;
}
