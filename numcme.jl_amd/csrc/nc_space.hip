// Device-resident sparse FSP state space.
//
// Replaces StateSpaceSparse (NumCME.jl src/statespace/sparse/sparsestatespace.jl) with a
// GPU open-addressing hash table. The reference's sequential semantics are kept exactly:
//
//  * expand! (sparsestatespace.jl:153-194) explores the explorable states last-first (its
//    Deque pop! takes from the back) and, within one state, reactions in list order. Here
//    every candidate gets its position in that sequential order; candidates are inserted
//    in parallel and a key's slot keeps the smallest position (atomicMin), so the first
//    occurrence wins as in _addstates! (:217-226). A prefix sum over the winners assigns
//    the reference's indices.
//  * The connectivity fill (:241-266) writes values that depend only on the final set of
//    states, so it runs one thread per (new state, reaction).
//  * deleteat! (:276-331) is a keep-flag scan, a compaction with index remapping, a hash
//    rebuild and a sink recomputation.
#include <atomic>
#include <type_traits>

#include "nc_space.h"

namespace nc {

namespace {

struct RList {
  int32_t n;
  int32_t r[kMaxReactions];
};

__global__ void k_fill_u32(uint32_t* p, int64_t n, uint32_t v) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    p[i] = v;
}

__global__ void k_table_insert_all(uint32_t* table, uint64_t mask, const int32_t* states, int ns, int64_t n) {
  int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= n) return;
  uint64_t h = hash_state(states + i * ns, ns) & mask;
  for (;;) {
    uint32_t old = atomicCAS(&table[h], HT_EMPTY, (uint32_t)i);
    if (old == HT_EMPTY) return;
    h = (h + 1) & mask;
  }
}

// Explorables of the first level: states with a sink on one of the listed reactions (and,
// when `select` is given, a nonzero select flag).
__global__ void k_flag_explorable(const uint32_t* sink_mask, int64_t n, uint32_t rmask, const uint32_t* select,
                                  uint32_t* flags) {
  int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i < n) flags[i] = ((sink_mask[i] & rmask) && (!select || select[i])) ? 1u : 0u;
}

__global__ void k_scatter_flagged(const uint32_t* flags, const uint32_t* ranks, int64_t n, int32_t* out) {
  int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i < n && flags[i]) out[ranks[i]] = (int32_t)i;
}

// Candidate `pos` in the reference's order: explorable E[nE-1-pos/|R'|] (LIFO), reaction
// R'[pos % |R'|]. `explorables == nullptr` means E[e] = base + e.
__global__ void k_gen_candidates(const int32_t* states, const int32_t* stoich, int ns, const int32_t* explorables,
                                 int64_t base, int64_t nE, RList rl, int32_t* cands) {
  int64_t pos = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (pos >= nE * rl.n) return;
  int64_t e = nE - 1 - pos / rl.n;
  int r = rl.r[pos % rl.n];
  int64_t src = explorables ? explorables[e] : base + e;
  for (int s = 0; s < ns; ++s) cands[pos * ns + s] = states[src * ns + s] + stoich[s + r * ns];
}

// A state's counts in registers: NS is at least the species count, so the loops unroll (a
// runtime count would put the array in scratch memory).
template <int NS>
struct Row {
  int32_t x[NS];
};
template <int NS>
__device__ inline Row<NS> load_row(const int32_t* p, int ns) {
  Row<NS> r;
#pragma unroll
  for (int s = 0; s < NS; ++s) r.x[s] = s < ns ? p[s] : 0;
  return r;
}
template <int NS>
__device__ inline bool row_nonneg(const Row<NS>& a) {
  bool ok = true;
#pragma unroll
  for (int s = 0; s < NS; ++s) ok = ok && a.x[s] >= 0;
  return ok;
}
template <int NS>
__device__ inline bool row_eq(const Row<NS>& a, const Row<NS>& b) {
  bool eq = true;
#pragma unroll
  for (int s = 0; s < NS; ++s) eq = eq && a.x[s] == b.x[s];
  return eq;
}
template <int NS>
__device__ inline uint64_t row_hash(const Row<NS>& a, int ns) {  // hash_state
  uint64_t h = 0x9E3779B97F4A7C15ull * (uint64_t)(ns + 1);
#pragma unroll
  for (int s = 0; s < NS; ++s)
    if (s < ns) h = mix64(h ^ (uint64_t)(uint32_t)a.x[s]);
  return h;
}
template <int NS, int SCOPE>
__device__ inline int32_t row_find(const uint32_t* table, uint64_t mask, const int32_t* states, int ns,
                                   const Row<NS>& x) {  // ht_find
  uint64_t h = row_hash<NS>(x, ns) & mask;
  for (;;) {
    const uint32_t v = __hip_atomic_load(&table[h], __ATOMIC_RELAXED, SCOPE);
    if (v == HT_EMPTY) return -1;
    if (!(v & HT_CAND) && row_eq<NS>(load_row<NS>(states + (int64_t)v * ns, ns), x)) return (int32_t)v;
    h = (h + 1) & mask;
  }
}
// Claim the slot of candidate `pos` with key x: its index, or -1 when x is in the space.
// Every tag ever stored in a slot belongs to the same key, so comparing against the one read
// is enough even if a smaller position replaces it concurrently. cand(p) is candidate p's key.
template <int NS, int SCOPE, class CAND>
__device__ inline int32_t row_claim(uint32_t* table, uint64_t mask, const int32_t* states, int ns, const Row<NS>& x,
                                    uint32_t pos, CAND cand) {
  const uint32_t tag = HT_CAND | pos;
  uint64_t h = row_hash<NS>(x, ns) & mask;
  for (;;) {
    uint32_t v = __hip_atomic_load(&table[h], __ATOMIC_RELAXED, SCOPE);
    if (v == HT_EMPTY) {
      uint32_t want = HT_EMPTY;
      if (__hip_atomic_compare_exchange_strong(&table[h], &want, tag, __ATOMIC_RELAXED, __ATOMIC_RELAXED, SCOPE))
        return (int32_t)h;
      v = want;
    }
    if (v & HT_CAND) {
      if (row_eq<NS>(cand(v & ~HT_CAND), x)) {
        __hip_atomic_fetch_min(&table[h], tag, __ATOMIC_RELAXED, SCOPE);
        return (int32_t)h;
      }
    } else if (row_eq<NS>(load_row<NS>(states + (int64_t)v * ns, ns), x)) {
      return -1;
    }
    h = (h + 1) & mask;
  }
}
// Connectivity of state idx along reaction r (sparsestatespace.jl:241-266)
template <int NS, int SCOPE>
__device__ inline void row_connect(const uint32_t* table, uint64_t mask, const int32_t* states, const int32_t* stoich,
                                   int ns, int nr, int64_t idx, int r, int32_t* state_conn, uint32_t* sink_mask) {
  const Row<NS> x = load_row<NS>(states + idx * ns, ns), d = load_row<NS>(stoich + r * ns, ns);
  Row<NS> y, z;
#pragma unroll
  for (int s = 0; s < NS; ++s) y.x[s] = x.x[s] - d.x[s], z.x[s] = x.x[s] + d.x[s];
  if (row_nonneg<NS>(y)) {
    const int32_t j = row_find<NS, SCOPE>(table, mask, states, ns, y);
    if (j >= 0) {
      state_conn[idx * nr + r] = j;
      __hip_atomic_fetch_and(&sink_mask[j], ~(1u << r), __ATOMIC_RELAXED, SCOPE);
    }
  }
  if (row_nonneg<NS>(z)) {
    const int32_t k = row_find<NS, SCOPE>(table, mask, states, ns, z);
    if (k < 0)
      __hip_atomic_fetch_or(&sink_mask[idx], 1u << r, __ATOMIC_RELAXED, SCOPE);
    else
      state_conn[(int64_t)k * nr + r] = (int32_t)idx;
  }
}

template <int NS>
__global__ void k_cand_insert(uint32_t* table, uint64_t mask, const int32_t* states, const int32_t* cands, int ns,
                              int64_t n_cand, int32_t* slot_of) {
  int64_t pos = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (pos >= n_cand) return;
  const Row<NS> x = load_row<NS>(cands + pos * ns, ns);
  // _is_all_nonnegative (sparsestatespace.jl:197-202)
  slot_of[pos] = !row_nonneg<NS>(x) ? -1
                                    : row_claim<NS, __HIP_MEMORY_SCOPE_AGENT>(
                                          table, mask, states, ns, x, (uint32_t)pos,
                                          [&](uint32_t p) { return load_row<NS>(cands + (int64_t)p * ns, ns); });
}

__global__ void k_first_flags(const uint32_t* table, const int32_t* slot_of, int64_t n_cand, uint32_t* flags) {
  int64_t pos = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (pos >= n_cand) return;
  int32_t sl = slot_of[pos];
  flags[pos] = (sl >= 0 && table[sl] == (HT_CAND | (uint32_t)pos)) ? 1u : 0u;
}

__global__ void k_commit(uint32_t* table, const int32_t* slot_of, const uint32_t* flags, const uint32_t* ranks,
                         const int32_t* cands, int ns, int nr, int64_t n_cand, int64_t n_old, int32_t* states,
                         int32_t* state_conn, uint32_t* sink_mask) {
  int64_t pos = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (pos >= n_cand || !flags[pos]) return;
  int64_t idx = n_old + ranks[pos];
  for (int s = 0; s < ns; ++s) states[idx * ns + s] = cands[pos * ns + s];
  for (int r = 0; r < nr; ++r) state_conn[idx * nr + r] = -1;
  sink_mask[idx] = 0u;
  table[slot_of[pos]] = (uint32_t)idx;
}

// Connectivity of the states [n_old, n_new).
template <int NS>
__global__ void k_connect_new(const uint32_t* table, uint64_t mask, const int32_t* states, const int32_t* stoich,
                              int ns, int nr, int64_t n_old, int64_t n_new, int32_t* state_conn,
                              uint32_t* sink_mask) {
  int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (t >= (n_new - n_old) * nr) return;
  row_connect<NS, __HIP_MEMORY_SCOPE_AGENT>(table, mask, states, stoich, ns, nr, n_old + t / nr, (int)(t % nr),
                                            state_conn, sink_mask);
}

// ---- levels with few candidates ---------------------------------------------------------
// A level of expansion is seven dependent launches and a synchronisation, 73 us however
// small it is. While a level has at most kSmallCands candidates, one workgroup runs level
// after level itself: the same passes separated by barriers, every atomic and every read
// of the table and the sink masks at workgroup scope. It stops when a level would have
// more, or when the rows or the table might not hold it, and says where.
constexpr int kSmallThreads = 1024;
constexpr int kSmallCands = 4096;
constexpr int kSmallPer = kSmallCands / kSmallThreads;
// A level costs a few dependent reads of the table per candidate and thread: an L2's latency
// up to here, beyond it memory's (the table of 2^20 states is 8 MB, an XCD's L2 holds 4).
// One workgroup against the launches, us a level: 30 and 68 on 251,000 states (501
// candidates), 75 and 90 on 501,000 (4,036), 60 and 64 on 1.0 million (1,001), 131 and 70 on
// 2.0 million (1,401). Candidates: 57 and 77 us at 4,860 on 5,456 states, 91 and 76 at 7,560.
constexpr int64_t kSmallStates = int64_t(1) << 19;
struct ExpandArgs {
  uint32_t* table;
  uint64_t mask;
  int32_t *states, *conn;
  uint32_t* sinks;
  const int32_t* stoich;
  int32_t* list;           // the first level's explorables: written here first when n_flag >= 0
  const uint32_t* select;  // flags, or null
  int32_t ns, nr, levels;
  uint32_t rmask;
  int32_t n_flag;  // >= 0: find the explorables among this many states (at most kSmallCands)
  int64_t n, base, nE, max_rows;
  RList rl;
  int64_t* out;  // pinned: levels done, states, first explorable, explorables, 1 if they are the list's
};

// Exclusive prefix sum over the workgroup in thread order, and the total; two barriers.
__device__ inline int small_scan(int v, int* s_wave, int* total) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int inc = v;
  for (int d = 1; d < 64; d <<= 1) {
    const int o = __shfl_up(inc, d, 64);
    if (lane >= d) inc += o;
  }
  if (lane == 63) s_wave[wave] = inc;
  __syncthreads();
  int before = 0, all = 0;
  for (int w = 0; w < kSmallThreads / 64; ++w) {
    const int x = s_wave[w];
    if (w < wave) before += x;
    all += x;
  }
  __syncthreads();
  *total = all;
  return before + inc - v;
}

template <int NS>
__global__ __launch_bounds__(kSmallThreads) void k_expand_small(ExpandArgs a) {
  constexpr int WG = __HIP_MEMORY_SCOPE_WORKGROUP;
  __shared__ int s_wave[kSmallThreads / 64];
  const int tid = threadIdx.x, ns = a.ns, nr = a.nr;
  int64_t n = a.n, base = a.base, nE = a.nE;
  const int32_t* list = a.list;
  if (a.n_flag >= 0) {
    int cnt = 0;
    uint32_t f = 0;
    for (int u = 0; u < kSmallPer; ++u) {
      const int i = tid * kSmallPer + u;
      if (i < a.n_flag && (a.sinks[i] & a.rmask) && (!a.select || a.select[i])) f |= 1u << u, ++cnt;
    }
    int total;
    int rank = small_scan(cnt, s_wave, &total);
    for (int u = 0; u < kSmallPer; ++u)
      if ((f >> u) & 1u) a.list[rank++] = tid * kSmallPer + u;
    nE = total;
    __syncthreads();
  }
  int level = 0;
  for (; level < a.levels; ++level) {
    const int64_t n_cand = nE * a.rl.n;
    if (n_cand == 0 || n_cand > kSmallCands || n + n_cand > a.max_rows) break;
    // candidate pos: explorable nE - 1 - pos / |R'| (last first), reaction R'[pos % |R'|]
    auto cand = [&](uint32_t pos) {
      const int64_t e = nE - 1 - pos / a.rl.n;
      const Row<NS> x = load_row<NS>(a.states + (list ? (int64_t)list[e] : base + e) * ns, ns),
                    d = load_row<NS>(a.stoich + a.rl.r[pos % a.rl.n] * ns, ns);
      Row<NS> y;
#pragma unroll
      for (int s = 0; s < NS; ++s) y.x[s] = x.x[s] + d.x[s];
      return y;
    };
    const int per = (int)((n_cand + kSmallThreads - 1) / kSmallThreads);
    int32_t slot[kSmallPer];
#pragma unroll
    for (int u = 0; u < kSmallPer; ++u) {
      slot[u] = -1;
      const int pos = tid * per + u;
      if (u < per && pos < n_cand) {
        const Row<NS> x = cand(pos);
        if (row_nonneg<NS>(x)) slot[u] = row_claim<NS, WG>(a.table, a.mask, a.states, ns, x, pos, cand);
      }
    }
    __syncthreads();
    int cnt = 0;
#pragma unroll
    for (int u = 0; u < kSmallPer; ++u) {
      // the slot's first occurrence keeps it
      if (slot[u] >= 0 && __hip_atomic_load(&a.table[slot[u]], __ATOMIC_RELAXED, WG) != (HT_CAND | (uint32_t)(tid * per + u)))
        slot[u] = -1;
      cnt += slot[u] >= 0;
    }
    int added;
    int64_t idx = n + small_scan(cnt, s_wave, &added);
#pragma unroll
    for (int u = 0; u < kSmallPer; ++u) {
      if (slot[u] < 0) continue;
      const Row<NS> x = cand(tid * per + u);
#pragma unroll
      for (int s = 0; s < NS; ++s)
        if (s < ns) a.states[idx * ns + s] = x.x[s];
      for (int r = 0; r < nr; ++r) a.conn[idx * nr + r] = -1;
      __hip_atomic_store(&a.sinks[idx], 0u, __ATOMIC_RELAXED, WG);
      __hip_atomic_store(&a.table[slot[u]], (uint32_t)idx, __ATOMIC_RELAXED, WG);
      ++idx;
    }
    __syncthreads();
    for (int t = tid; t < added * nr; t += kSmallThreads)
      row_connect<NS, WG>(a.table, a.mask, a.states, a.stoich, ns, nr, n + t / nr, t % nr, a.conn, a.sinks);
    __syncthreads();
    // the next level explores the states just added, in ascending order
    list = nullptr;
    base = n;
    nE = added;
    n += added;
  }
  if (tid == 0) {
    a.out[0] = level;
    a.out[1] = n;
    a.out[2] = base;
    a.out[3] = nE;
    a.out[4] = list ? 1 : 0;
  }
}

__global__ void k_mark_ids(const int64_t* ids, int64_t m, uint32_t* keep) {
  int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i < m) keep[ids[i]] = 0u;
}

__global__ void k_compact(const uint32_t* keep, const uint32_t* ranks, int64_t n, int ns, int nr, const int32_t* states,
                          const int32_t* state_conn, const uint32_t* sink_mask, int32_t* states2, int32_t* conn2,
                          uint32_t* sink2) {
  int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= n || !keep[i]) return;
  int64_t d = ranks[i];
  for (int s = 0; s < ns; ++s) states2[d * ns + s] = states[i * ns + s];
  for (int r = 0; r < nr; ++r) {
    int32_t c = state_conn[i * nr + r];
    conn2[d * nr + r] = (c >= 0 && keep[c]) ? (int32_t)ranks[c] : -1;
  }
  sink2[d] = sink_mask[i];
}

// sparsestatespace.jl:318-329: new sinks for states whose successor was deleted.
__global__ void k_recompute_sinks(const uint32_t* table, uint64_t mask, const int32_t* states, const int32_t* stoich,
                                  int ns, int nr, int64_t n, uint32_t* sink_mask) {
  int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= n) return;
  uint32_t m = sink_mask[i];
  int32_t z[kMaxSpecies];
  for (int r = 0; r < nr; ++r) {
    if (m & (1u << r)) continue;
    bool ok = true;
    for (int s = 0; s < ns; ++s) {
      z[s] = states[i * ns + s] + stoich[s + r * ns];
      ok = ok && z[s] >= 0;
    }
    if (ok && ht_find(table, mask, states, ns, z) < 0) m |= 1u << r;
  }
  sink_mask[i] = m;
}

__global__ void k_lookup(const uint32_t* table, uint64_t mask, const int32_t* states, int ns, const int32_t* q,
                         int64_t nq, int64_t* out) {
  int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= nq) return;
  int32_t x[kMaxSpecies];
  bool ok = true;
  for (int s = 0; s < ns; ++s) {
    x[s] = q[i * ns + s];
    ok = ok && x[s] >= 0;
  }
  out[i] = (ok && mask) ? (int64_t)ht_find(table, mask, states, ns, x) : -1;
}

constexpr int kBlock = 256;

// f with the kernels' species count as a constant: the next of 1, 2, 3, 4, 6, 8, 16
template <class F>
void by_species(int ns, F&& f) {
  if (ns <= 1)
    f(std::integral_constant<int, 1>{});
  else if (ns == 2)
    f(std::integral_constant<int, 2>{});
  else if (ns == 3)
    f(std::integral_constant<int, 3>{});
  else if (ns == 4)
    f(std::integral_constant<int, 4>{});
  else if (ns <= 6)
    f(std::integral_constant<int, 6>{});
  else if (ns <= 8)
    f(std::integral_constant<int, 8>{});
  else
    f(std::integral_constant<int, kMaxSpecies>{});
}

}  // namespace

void space_reserve(nc_space_s* sp, int64_t rows) {
  if (rows <= sp->cap) return;
  int64_t cap = sp->cap ? sp->cap : 1024;
  while (cap < rows) cap *= 2;
  sp->states.grow_keep((size_t)cap * sp->ns, (size_t)sp->n * sp->ns, sp->stream.s);
  sp->state_conn.grow_keep((size_t)cap * sp->nr, (size_t)sp->n * sp->nr, sp->stream.s);
  sp->sink_mask.grow_keep((size_t)cap, (size_t)sp->n, sp->stream.s);
  sp->cap = cap;
}

void space_rebuild_table(nc_space_s* sp, int64_t min_entries) {
  uint64_t cap = 1024;
  while (cap < 2 * (uint64_t)min_entries) cap *= 2;
  NC_REQUIRE(cap <= (1ull << 31), NC_ERR_OVERFLOW, "state space too large for the hash table");
  if (cap > sp->table_cap || !sp->table.p) {
    sp->table.alloc(cap);
    sp->table_cap = cap;
  }
  hipStream_t s = sp->stream.s;
  k_fill_u32<<<grid_for(sp->table_cap, kBlock), kBlock, 0, s>>>(sp->table.p, (int64_t)sp->table_cap, HT_EMPTY);
  if (sp->n)
    k_table_insert_all<<<grid_for(sp->n, kBlock), kBlock, 0, s>>>(sp->table.p, sp->table_cap - 1, sp->states.p,
                                                                   sp->ns, sp->n);
  NC_CHECK_HIP(hipGetLastError());
}

// Deduplicate and append the n_cand candidates held in sp->cands (candidate order is the
// reference's _addstates! order), then fill connectivity for the new states.
void space_add_candidates(nc_space_s* sp, int64_t n_cand) {
  if (n_cand <= 0) return;
  hipStream_t s = sp->stream.s;
  NC_REQUIRE(sp->n + n_cand < (int64_t)0x7FFFFFF0, NC_ERR_OVERFLOW, "state space exceeds 2^31 states");
  space_reserve(sp, sp->n + n_cand);
  if ((uint64_t)(2 * (sp->n + n_cand)) > sp->table_cap) space_rebuild_table(sp, sp->n + n_cand);
  sp->slot_of.reserve(n_cand);
  sp->flags.reserve(n_cand);
  sp->ranks.reserve(n_cand);
  const uint64_t mask = sp->table_cap - 1;
  by_species(sp->ns, [&](auto NS) {
    k_cand_insert<NS.value><<<grid_for(n_cand, kBlock), kBlock, 0, s>>>(sp->table.p, mask, sp->states.p, sp->cands.p,
                                                                        sp->ns, n_cand, sp->slot_of.p);
  });
  k_first_flags<<<grid_for(n_cand, kBlock), kBlock, 0, s>>>(sp->table.p, sp->slot_of.p, n_cand, sp->flags.p);
  NC_CHECK_HIP(hipGetLastError());
  uint32_t added = 0;
  exclusive_scan_u32(sp->flags.p, sp->ranks.p, n_cand, sp->scan_tmp, s, &added);
  const int64_t n_old = sp->n;
  k_commit<<<grid_for(n_cand, kBlock), kBlock, 0, s>>>(sp->table.p, sp->slot_of.p, sp->flags.p, sp->ranks.p,
                                                        sp->cands.p, sp->ns, sp->nr, n_cand, n_old, sp->states.p,
                                                        sp->state_conn.p, sp->sink_mask.p);
  NC_CHECK_HIP(hipGetLastError());
  sp->n = n_old + added;
  if (added) {
    int64_t work = (int64_t)added * sp->nr;
    by_species(sp->ns, [&](auto NS) {
      k_connect_new<NS.value><<<grid_for(work, kBlock), kBlock, 0, s>>>(sp->table.p, mask, sp->states.p, sp->d_stoich.p,
                                                                        sp->ns, sp->nr, n_old, sp->n,
                                                                        sp->state_conn.p, sp->sink_mask.p);
    });
    NC_CHECK_HIP(hipGetLastError());
    sp->version++;
  }
}

static void space_expand(nc_space_s* sp, int levels, const std::vector<int32_t>& rlist,
                         const uint32_t* select = nullptr) {
  if (levels <= 0) return;  // sparsestatespace.jl:154-156
  hipStream_t s = sp->stream.s;
  RList rl{};
  rl.n = (int32_t)rlist.size();
  uint32_t rmask = 0;
  for (int k = 0; k < rl.n; ++k) {
    rl.r[k] = rlist[k];
    rmask |= 1u << rlist[k];
  }
  // first-level explorables: ascending indices with a sink on some listed reaction (:165-173)
  int64_t nE = 0, base = 0;
  const int32_t* E = nullptr;
  int level = 0;
  if (sp->n == 0 || rl.n == 0) return;
  sp->explorables.reserve(std::max<int64_t>(sp->n, kSmallCands));
  E = sp->explorables.p;
  bool listed = sp->n > kSmallCands;  // a small space's explorables are found by the small levels
  if (listed) {
    sp->flags.reserve(sp->n);
    sp->ranks.reserve(sp->n);
    k_flag_explorable<<<grid_for(sp->n, kBlock), kBlock, 0, s>>>(sp->sink_mask.p, sp->n, rmask, select,
                                                                   sp->flags.p);
    uint32_t cnt = 0;
    exclusive_scan_u32(sp->flags.p, sp->ranks.p, sp->n, sp->scan_tmp, s, &cnt);
    k_scatter_flagged<<<grid_for(sp->n, kBlock), kBlock, 0, s>>>(sp->flags.p, sp->ranks.p, sp->n, sp->explorables.p);
    NC_CHECK_HIP(hipGetLastError());
    nE = cnt;
  }
  while (level < levels) {  // :176-192
    if (!listed || (nE > 0 && nE * rl.n <= kSmallCands && sp->n <= kSmallStates)) {
      // room for several such levels, so that the kernel rarely stops for want of it
      const int64_t room = sp->n + (int64_t)kSmallCands * std::min(levels - level, 8);
      space_reserve(sp, room);
      if ((uint64_t)(2 * room) > sp->table_cap) space_rebuild_table(sp, room);
      ExpandArgs a{};
      a.table = sp->table.p;
      a.mask = sp->table_cap - 1;
      a.states = sp->states.p;
      a.conn = sp->state_conn.p;
      a.sinks = sp->sink_mask.p;
      a.stoich = sp->d_stoich.p;
      a.list = E ? sp->explorables.p : nullptr;
      a.select = select;
      a.ns = sp->ns;
      a.nr = sp->nr;
      a.levels = levels - level;
      a.rmask = rmask;
      a.n_flag = listed ? -1 : (int32_t)sp->n;
      a.n = sp->n;
      a.nE = nE;
      a.base = base;
      a.max_rows = std::min<int64_t>(sp->cap, (int64_t)(sp->table_cap / 2));
      a.rl = rl;
      int64_t* out = static_cast<int64_t*>(host_stage(6));
      NC_CHECK_HIP(hipHostGetDevicePointer(reinterpret_cast<void**>(&a.out), out, 0));
      by_species(sp->ns, [&](auto NS) { k_expand_small<NS.value><<<1, kSmallThreads, 0, s>>>(a); });
      NC_CHECK_HIP(hipGetLastError());
      NC_CHECK_HIP(hipStreamSynchronize(s));
      level += (int)out[0];
      if (out[1] > sp->n) sp->version++;
      sp->n = out[1];
      base = out[2];
      nE = out[3];
      if (!out[4]) E = nullptr;
      listed = true;
      if (nE == 0) break;
      if (out[0] > 0) continue;  // stopped for rows (or done): the next round makes room
    }
    const int64_t n_cand = nE * rl.n;
    if (n_cand == 0 || level >= levels) break;
    NC_REQUIRE(n_cand < (int64_t)0x7FFFFFF0, NC_ERR_OVERFLOW, "too many expansion candidates");
    sp->cands.reserve((size_t)n_cand * sp->ns);
    k_gen_candidates<<<grid_for(n_cand, kBlock), kBlock, 0, s>>>(sp->states.p, sp->d_stoich.p, sp->ns, E, base, nE,
                                                                  rl, sp->cands.p);
    NC_CHECK_HIP(hipGetLastError());
    const int64_t n_old = sp->n;
    space_add_candidates(sp, n_cand);
    // the next level explores the states just added, in ascending order (:189-191)
    E = nullptr;
    base = n_old;
    nE = sp->n - n_old;
    ++level;
  }
}

__global__ void k_compact_vec(const uint32_t* keep, const uint32_t* ranks, int64_t n, const double* in, double* out) {
  int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i < n && keep[i]) out[ranks[i]] = in[i];
}

// deleteat! with the (sorted, unique, in-range) ids already on the device. The vectors
// vin[k] (length n before the call) are compacted the same way into vout[k].
void space_delete_device(nc_space_s* sp, const int64_t* d_ids, int64_t m, int nvec, const double* const* vin,
                         double* const* vout) {
  hipStream_t s = sp->stream.s;
  if (sp->n == 0) return;
  const int64_t n = sp->n;
  sp->flags.reserve(n);
  sp->ranks.reserve(n);
  k_fill_u32<<<grid_for(n, kBlock), kBlock, 0, s>>>(sp->flags.p, n, 1u);
  if (m) k_mark_ids<<<grid_for(m, kBlock), kBlock, 0, s>>>(d_ids, m, sp->flags.p);
  uint32_t kept = 0;
  exclusive_scan_u32(sp->flags.p, sp->ranks.p, n, sp->scan_tmp, s, &kept);
  for (int k = 0; k < nvec; ++k)
    k_compact_vec<<<grid_for(n, kBlock), kBlock, 0, s>>>(sp->flags.p, sp->ranks.p, n, vin[k], vout[k]);
  DevBuf<int32_t> st2((size_t)sp->cap * sp->ns), cn2((size_t)sp->cap * sp->nr);
  DevBuf<uint32_t> sk2((size_t)sp->cap);
  k_compact<<<grid_for(n, kBlock), kBlock, 0, s>>>(sp->flags.p, sp->ranks.p, n, sp->ns, sp->nr, sp->states.p,
                                                    sp->state_conn.p, sp->sink_mask.p, st2.p, cn2.p, sk2.p);
  NC_CHECK_HIP(hipGetLastError());
  NC_CHECK_HIP(hipStreamSynchronize(s));
  sp->states = std::move(st2);
  sp->state_conn = std::move(cn2);
  sp->sink_mask = std::move(sk2);
  sp->n = kept;
  sp->version++;
  if (sp->n == 0) return;  // :306-308
  space_rebuild_table(sp, sp->n);
  k_recompute_sinks<<<grid_for(sp->n, kBlock), kBlock, 0, s>>>(sp->table.p, sp->table_cap - 1, sp->states.p,
                                                                sp->d_stoich.p, sp->ns, sp->nr, sp->n,
                                                                sp->sink_mask.p);
  NC_CHECK_HIP(hipGetLastError());
}

static void space_delete(nc_space_s* sp, int64_t m, const int64_t* ids_host) {
  for (int64_t k = 0; k < m; ++k) {
    NC_REQUIRE(ids_host[k] >= 0 && ids_host[k] < sp->n, NC_ERR_ARG, "deleteat!: index out of range");
    NC_REQUIRE(k == 0 || ids_host[k] > ids_host[k - 1], NC_ERR_ARG, "deleteat!: indices must be unique and sorted");
  }
  if (sp->n == 0) return;
  DevBuf<int64_t> d_ids(m ? m : 1);
  if (m) NC_CHECK_HIP(hipMemcpyAsync(d_ids.p, ids_host, m * sizeof(int64_t), hipMemcpyHostToDevice, sp->stream.s));
  space_delete_device(sp, d_ids.p, m, 0, nullptr, nullptr);
}

nc_space_s* space_create(int ns, int nr, const int32_t* stoich, int64_t n_init, const int32_t* init_states) {
  NC_REQUIRE(ns >= 1 && ns <= kMaxSpecies, NC_ERR_UNSUPPORTED, "species count must be in 1..16");
  NC_REQUIRE(nr >= 1 && nr <= kMaxReactions, NC_ERR_UNSUPPORTED, "reaction count must be in 1..32");
  NC_REQUIRE(stoich, NC_ERR_ARG, "null stoichiometry matrix");
  NC_REQUIRE(n_init >= 0 && (n_init == 0 || init_states), NC_ERR_ARG, "bad initial state list");
  int dev_count = 0;
  if (hipGetDeviceCount(&dev_count) != hipSuccess || dev_count == 0)
    throw Error(NC_ERR_NO_DEVICE, "no HIP device available");
  auto sp = new nc_space_s();
  static std::atomic<uint64_t> next_uid{1};
  sp->uid = next_uid++;
  try {
    sp->ns = ns;
    sp->nr = nr;
    sp->stoich.assign(stoich, stoich + (size_t)ns * nr);
    sp->d_stoich.alloc((size_t)ns * nr);
    // on the space's stream from its own host copy (the constructor ends with a
    // synchronisation of that stream)
    NC_CHECK_HIP(hipMemcpyAsync(sp->d_stoich.p, sp->stoich.data(), sizeof(int32_t) * ns * nr, hipMemcpyHostToDevice,
                                sp->stream.s));
    space_reserve(sp, std::max<int64_t>(n_init, 1));
    space_rebuild_table(sp, std::max<int64_t>(n_init, 1));
    if (n_init) {
      sp->cands.reserve((size_t)n_init * ns);
      NC_CHECK_HIP(hipMemcpyAsync(sp->cands.p, init_states, sizeof(int32_t) * ns * n_init, hipMemcpyHostToDevice,
                                  sp->stream.s));
      space_add_candidates(sp, n_init);  // _addstates!(space, initstates): :122
    }
    NC_CHECK_HIP(hipStreamSynchronize(sp->stream.s));
  } catch (...) {
    delete sp;
    throw;
  }
  return sp;
}

void space_expand_list(nc_space_s* sp, int levels, const std::vector<int32_t>& rlist, const uint32_t* select) {
  space_expand(sp, levels, rlist, select);
}

}  // namespace nc

using namespace nc;

extern "C" {

int nc_space_create(int32_t ns, int32_t nr, const int32_t* stoich, int64_t n_init, const int32_t* init_states,
                    nc_space* out) {
  return guard([&] {
    NC_REQUIRE(out, NC_ERR_ARG, "null output handle");
    *out = space_create(ns, nr, stoich, n_init, init_states);
  });
}

int nc_space_destroy(nc_space sp) {
  return guard([&] { delete sp; });
}

int nc_space_expand(nc_space sp, int32_t levels, int32_t n_only, const int32_t* only) {
  return guard([&] {
    NC_REQUIRE(sp, NC_ERR_ARG, "null space");
    std::vector<int32_t> rl;
    if (n_only > 0) {
      NC_REQUIRE(only, NC_ERR_ARG, "null reaction list");
      NC_REQUIRE(n_only <= kMaxReactions, NC_ERR_ARG, "reaction list too long");
      for (int k = 0; k < n_only; ++k) {
        NC_REQUIRE(only[k] >= 0 && only[k] < sp->nr, NC_ERR_ARG, "reaction index out of range");
        rl.push_back(only[k]);
      }
    } else {
      for (int r = 0; r < sp->nr; ++r) rl.push_back(r);  // isempty(onlyreactions) -> all (:163)
    }
    space_expand(sp, levels, rl);
    NC_CHECK_HIP(hipStreamSynchronize(sp->stream.s));
  });
}

int nc_space_delete(nc_space sp, int64_t m, const int64_t* ids) {
  return guard([&] {
    NC_REQUIRE(sp, NC_ERR_ARG, "null space");
    NC_REQUIRE(m >= 0 && (m == 0 || ids), NC_ERR_ARG, "bad id list");
    space_delete(sp, m, ids);
    NC_CHECK_HIP(hipStreamSynchronize(sp->stream.s));
  });
}

int nc_space_count(nc_space sp, int64_t* n, int32_t* nsinks) {
  return guard([&] {
    NC_REQUIRE(sp, NC_ERR_ARG, "null space");
    if (n) *n = sp->n;
    if (nsinks) *nsinks = sp->nr;
  });
}

int nc_space_get_states(nc_space sp, int32_t* out) {
  return guard([&] {
    NC_REQUIRE(sp && (out || sp->n == 0), NC_ERR_ARG, "null argument");
    if (sp->n)
      NC_CHECK_HIP(hipMemcpy(out, sp->states.p, sizeof(int32_t) * sp->n * sp->ns, hipMemcpyDeviceToHost));
  });
}

int nc_space_get_state_conn(nc_space sp, int32_t* out) {
  return guard([&] {
    NC_REQUIRE(sp && (out || sp->n == 0), NC_ERR_ARG, "null argument");
    if (sp->n)
      NC_CHECK_HIP(hipMemcpy(out, sp->state_conn.p, sizeof(int32_t) * sp->n * sp->nr, hipMemcpyDeviceToHost));
  });
}

int nc_space_get_sink_conn(nc_space sp, int32_t* out) {
  return guard([&] {
    NC_REQUIRE(sp && (out || sp->n == 0), NC_ERR_ARG, "null argument");
    if (!sp->n) return;
    std::vector<uint32_t> m(sp->n);
    NC_CHECK_HIP(hipMemcpy(m.data(), sp->sink_mask.p, sizeof(uint32_t) * sp->n, hipMemcpyDeviceToHost));
    for (int64_t i = 0; i < sp->n; ++i)
      for (int r = 0; r < sp->nr; ++r) out[i * sp->nr + r] = (m[i] >> r) & 1u ? r : -1;
  });
}

int nc_space_lookup(nc_space sp, int64_t n, const int32_t* q, int64_t* out) {
  return guard([&] {
    NC_REQUIRE(sp && n >= 0 && (n == 0 || (q && out)), NC_ERR_ARG, "null argument");
    if (n == 0) return;
    hipStream_t s = sp->stream.s;
    DevBuf<int32_t> dq((size_t)n * sp->ns);
    DevBuf<int64_t> dout((size_t)n);
    NC_CHECK_HIP(hipMemcpyAsync(dq.p, q, sizeof(int32_t) * n * sp->ns, hipMemcpyHostToDevice, s));
    k_lookup<<<grid_for(n, kBlock), kBlock, 0, s>>>(sp->table.p, sp->n ? sp->table_cap - 1 : 0, sp->states.p, sp->ns,
                                                     dq.p, n, dout.p);
    NC_CHECK_HIP(hipGetLastError());
    NC_CHECK_HIP(hipMemcpyAsync(out, dout.p, sizeof(int64_t) * n, hipMemcpyDeviceToHost, s));
    NC_CHECK_HIP(hipStreamSynchronize(s));
  });
}

}  // extern "C"
