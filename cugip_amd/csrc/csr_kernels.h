// The generic-graph solve as one kernel (gfx950, wave64). Included by csr_solver.hip only.
//
// Push-relabel on an irregular graph is a chain of some hundreds to thousands of dependent steps (BFS
// levels, push steps), each a short gather: what bounds it is the latency of a step, not bytes. So the
// whole solve runs in one launch whose steps are separated by a barrier over few, large workgroups
// (2-3 us at 64 workgroups of 1024 threads, against a launch and a host read of about 16 us per
// level before), and a step whose list is short is run by workgroup 0 alone between workgroup barriers.
// Measured (lattice-like graphs of 7.8 arcs a vertex): 1 M vertices 267 -> 25 ms, 19683 vertices
// 22.3 -> 2.0 ms; a step of 1 M vertices' solve takes 9 us up to 4096 list entries and 22 us at 16-64 K.
//
// Between two relabels the push is synchronous push/relabel: every step takes each vertex that
// holds excess, pushes along its admissible arcs (neighbour exactly one label lower) and raises
// the label of a vertex whose admissible arcs are all saturated. One step is one phase, without
// a barrier between push and relabel; labels stay valid (h(v) <= h(u) + 1 over every open arc v -> u):
//   * u -> v and v -> u are never pushed in the same step (a pusher uses its label from before the
//     step, and labels only rise), so a pair's residuals have one writer per step;
//   * a push w -> v opens v -> w while v may be raising its label without having seen it. w's label is
//     above v's then, and w -> v was open, so v's new label is held to h(w) + 1 for every neighbour w
//     with a higher label and an open arc w -> v, whether it pushes or not.
// With valid labels distances to t never fall, so the rounds of exact BFS relabels end as those of
// any push-relabel.
//
// Data: arc a of vertex v has ends[a] = {head, mate} and pair[a] = {residual of a, residual of its
// mate}. Both directions are kept at both arcs, so the BFS (which needs the residual towards v) reads
// an arc's own record instead of gathering its mate's, and a push writes both records without
// reading the mate's. The lanes of a group (kGroup of a wave) share a vertex and read its arcs side
// by side.
#pragma once

#include "common.h"
#include "csr_control.h"

namespace cgp {

constexpr int kCsrThreads = 1024;
constexpr int kCsrWaves = kCsrThreads / 64;
constexpr int kCsrStage = 4096;      // list entries a workgroup collects in LDS per step
constexpr int kCsrMinSteps = 16;     // push steps after a relabel: twice its levels, at least this
constexpr long long kCsrGatherTicks = 25000000;  // wait for the launch's workgroups (100 MHz): 0.25 s

struct CsrArgs {
	int n;
	const int32_t *first;
	const int2 *ends;
	int2 *pair;
	int32_t *e, *rt, *h, *mark;
	int32_t *queue, *list[2];
	int32_t *starts;  // n + 2: queue end after each level
	CsrControl *ctl;
	int32_t max_rounds;
	int32_t stages;
	int32_t solo_limit;  // list length that workgroup 0 runs alone
};

// List entries of a workgroup, collected in LDS and stored by one reservation per step. (An atomic
// per wave on one word serialises in the L2, about 12 ns each: over a level of 50000 vertices
// that was most of the level's time.)
struct CsrStageBuffer {
	int32_t count, base;
	int32_t entry[kCsrStage];
};

struct CsrShared {
	CsrStageBuffer next, active;
	unsigned long long seen;
	int32_t gate;
	long long red[kCsrWaves];
};

// What a workgroup knows of the running phase.
struct CsrPhase {
	unsigned index;
	bool solo;  // no other workgroup takes part
};

__device__ inline unsigned long long *phase_word(const CsrArgs &g, const CsrPhase &ph)
{
	return &g.ctl->word[ph.index % 3u];
}

// Where a step's entries go: a list under construction and the word that reserves places in it. A
// workgroup that is the list's only writer needs no reservation (direct).
struct CsrList {
	int32_t *at;
	unsigned long long *word;  // entries in the high half (the phase word)
	int32_t *counter;          // or a plain count
	bool direct;
	__device__ int32_t reserve(int32_t entries) const
	{
		return word ? (int32_t)(atomicAdd(word, (unsigned long long)entries << 32) >> 32)
		            : atomicAdd(counter, entries);
	}
};

// Appends value where pred holds (all lanes of the wave take part). Entries beyond the LDS stage
// are stored at once, with one reservation per wave.
__device__ inline void stage_append(CsrStageBuffer &st, bool pred, int32_t value, const CsrList &list)
{
	const unsigned long long mask = __ballot(pred);
	if (!mask) {
		return;
	}
	const int lane = threadIdx.x & 63;
	const int entries = (int)__popcll(mask);
	int32_t base = 0;
	if (lane == 0) {
		base = atomicAdd(&st.count, entries);
	}
	base = __builtin_amdgcn_readfirstlane(base);
	const int32_t p = base + (int)__popcll(mask & ((1ull << lane) - 1ull));
	if (pred && p < kCsrStage) {
		st.entry[p] = value;
	}
	if (base + entries > kCsrStage) {  // (the same for the whole wave)
		const int32_t from = base > kCsrStage ? base : kCsrStage;
		int32_t place = from;
		if (!list.direct) {
			if (lane == 0) {
				place = list.reserve(base + entries - from);
			}
			place = __builtin_amdgcn_readfirstlane(place);
		}
		if (pred && p >= kCsrStage) {
			list.at[place + (p - from)] = value;
		}
	}
}

// Stores the staged entries (after the last append) and empties the stage. Returns the entries of
// this workgroup, those already stored among them.
__device__ inline int32_t stage_flush(CsrStageBuffer &st, const CsrList &list)
{
	__syncthreads();
	const int32_t total = st.count;
	const int32_t staged = total < kCsrStage ? total : kCsrStage;
	if (total > 0) {  // (the same for the whole workgroup)
		int32_t base = 0;
		if (!list.direct) {
			if (threadIdx.x == 0) {
				st.base = list.reserve(staged);
			}
			__syncthreads();
			base = st.base;
		}
		for (int i = threadIdx.x; i < staged; i += kCsrThreads) {
			list.at[base + i] = st.entry[i];
		}
		__syncthreads();
		if (threadIdx.x == 0) {
			st.count = 0;
		}
	}
	return total;
}

// End of a phase over the grid. Returns the entries appended during it (by all workgroups). All stores
// of the phase are visible to every workgroup afterwards.
__device__ inline int32_t grid_phase_end(const CsrArgs &g, CsrShared &sh, CsrPhase &ph)
{
	// every wave's stores have reached the L2 before thread 0 writes the L2 back and arrives
	__builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
	__builtin_amdgcn_s_waitcnt(0);
	__syncthreads();
	if (threadIdx.x == 0) {
		unsigned long long *word = phase_word(g, ph);
		if (blockIdx.x == 0) {
			// the next phase's word (last read two barriers ago)
			__hip_atomic_store(&g.ctl->word[(ph.index + 1u) % 3u], 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
		}
		__builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
		__hip_atomic_fetch_add(word, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
		unsigned long long seen;
		while ((uint32_t)(seen = __hip_atomic_load(word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) < gridDim.x) {
			__builtin_amdgcn_s_sleep(1);
		}
		__builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
		sh.seen = seen;
	}
	__syncthreads();
	++ph.index;
	return (int32_t)(sh.seen >> 32);
}

// Before the first barrier: whether every workgroup of the launch is running. The barriers need that
// (a workgroup that waits for a place on a CU held by one that waits for it would wait for ever),
// and an ordinary launch does not promise it when other kernels that wait fill the chip. The last
// workgroup to arrive opens the launch; a workgroup that waited kCsrGatherTicks closes it instead,
// and every workgroup, those that start later too, leaves without having changed anything. Once
// all are running they stay so until they end. (A cooperative launch would promise it, but a second
// process on the same GPU is refused one.)
__device__ inline bool all_running(const CsrArgs &g, CsrShared &sh)
{
	if (threadIdx.x == 0) {
		int32_t *gate = &g.ctl->gate;
		if (atomicAdd(&g.ctl->arrived, 1) == (int)gridDim.x - 1) {
			atomicCAS(gate, 0, kCsrGateOpen);
		}
		const long long begun = wall_clock64();
		int32_t state;
		while ((state = __hip_atomic_load(gate, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) == 0) {
			__builtin_amdgcn_s_sleep(8);
			if (wall_clock64() - begun > kCsrGatherTicks) {
				atomicCAS(gate, 0, kCsrGateClosed);
			}
		}
		sh.gate = state;
	}
	__syncthreads();
	return sh.gate == kCsrGateOpen;
}

// The list that a step appends to, starting at `at`.
__device__ inline CsrList step_list(const CsrArgs &g, const CsrPhase &ph, int32_t *at)
{
	return CsrList{at, ph.solo ? nullptr : phase_word(g, ph), nullptr, ph.solo};
}

// End of a step: the staged entries are stored to its list, and the number of entries that the step
// appended is returned. A workgroup that runs alone only needs its own barriers.
__device__ inline int32_t step_end(const CsrArgs &g, CsrShared &sh, CsrPhase &ph, const CsrList &list)
{
	const int32_t own = stage_flush(sh.next, list);
	if (ph.solo) {
		__syncthreads();
		return own;
	}
	return grid_phase_end(g, sh, ph);
}

// First list entry of this wave and the distance to its next ones: waves take kPer consecutive
// entries, dealt out over the workgroups first, so that a short list spreads over all of them.
template <int kPer>
__device__ inline void wave_share(const CsrPhase &ph, int &begin, int &stride)
{
	const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
	const int blocks = ph.solo ? 1 : (int)gridDim.x;
	const int block = ph.solo ? 0 : (int)blockIdx.x;
	begin = (wave * blocks + block) * kPer;
	stride = kCsrWaves * blocks * kPer;
}

// Start of a search: labels (or marks) of every vertex, the seeds into the queue. A relabel also
// appends the vertices with excess that it reaches to the active list.
template <bool kClosure>
__device__ inline void search_seed(const CsrArgs &g, CsrShared &sh, const CsrPhase &ph, int32_t threshold,
                                   const CsrList &queue, const CsrList &active)
{
	int begin, stride;
	wave_share<64>(ph, begin, stride);
	for (int64_t base = begin; base < g.n; base += stride) {
		const int64_t v = base + (threadIdx.x & 63);
		bool seed = false, holds = false;
		if (v < g.n) {
			if (kClosure) {
				seed = g.e[v] > 0;
				g.mark[v] = seed ? 1 : 0;
			} else {
				seed = g.rt[v] > threshold;
				holds = seed && g.e[v] > 0;
				g.h[v] = seed ? 1 : kLabelInf;
			}
		}
		stage_append(sh.next, seed, (int32_t)v, queue);
		if (!kClosure) {
			stage_append(sh.active, holds, (int32_t)v, active);
		}
	}
}

// One level: the unvisited neighbours u of the frontier queue[qs, qe) that can reach it (relabel:
// residual u -> v > threshold) or that it reaches (closure: residual v -> u > 0).
template <int kGroup, bool kClosure>
__device__ inline void search_level(const CsrArgs &g, CsrShared &sh, const CsrPhase &ph, int qs, int qe, int32_t level,
                                    int32_t threshold, const CsrList &queue, const CsrList &active)
{
	constexpr int kPer = 64 / kGroup;
	const int sub = threadIdx.x % kGroup, slot = (threadIdx.x & 63) / kGroup;
	int32_t *visited = kClosure ? g.mark : g.h;
	const int32_t fresh = kClosure ? 0 : kLabelInf;
	int begin, stride;
	wave_share<kPer>(ph, begin, stride);
	const int count = qe - qs;
	for (int64_t base = begin; base < count; base += stride) {
		uint32_t a = 0, end = 0;
		if (base + slot < count) {
			const int v = g.queue[qs + (int)base + slot];
			a = (uint32_t)g.first[v] + sub;
			end = (uint32_t)g.first[v + 1];
		}
		while (__any(a < end)) {
			bool claimed = false, holds = false;
			int u = 0;
			if (a < end) {
				u = g.ends[a].x;
				const int2 p = g.pair[a];
				if ((kClosure ? p.x > 0 : p.y > threshold) && visited[u] == fresh) {
					claimed = atomicCAS(&visited[u], fresh, kClosure ? 1 : level + 1) == fresh;
					holds = !kClosure && claimed && g.e[u] > 0;
				}
				a += kGroup;
			}
			stage_append(sh.next, claimed, u, queue);
			if (!kClosure) {
				stage_append(sh.active, holds, u, active);
			}
		}
	}
}

// One synchronous push/relabel step over in[0, count); the vertices that hold excess after it (and
// have a finite label) are appended to out, each once: a vertex of the list by itself when excess
// is left, any other by the push that made its excess positive.
template <int kGroup>
__device__ inline void push_step(const CsrArgs &g, CsrShared &sh, const CsrPhase &ph, const int32_t *in, int count,
                                 const CsrList &out, int32_t threshold, long long &sink)
{
	constexpr int kPer = 64 / kGroup;
	const int sub = threadIdx.x % kGroup, slot = (threadIdx.x & 63) / kGroup;
	int begin, stride;
	wave_share<kPer>(ph, begin, stride);
	for (int64_t base = begin; base < count; base += stride) {
		int v = -1;
		uint32_t at = 0, end = 0;       // next arcs of the group
		int32_t x = 0, x0 = 0, hv = 0;  // excess left and at the start, label: the same in a group
		if (base + slot < count) {
			v = in[base + slot];
			at = (uint32_t)g.first[v];
			end = (uint32_t)g.first[v + 1];
			x0 = x = g.e[v];
			hv = g.h[v];
			const int32_t rtv = g.rt[v];
			const int32_t fs = x < rtv ? x : rtv;
			if (fs > 0) {
				x -= fs;
				if (sub == 0) {
					g.rt[v] = rtv - fs;
					sink += fs;
				}
			}
		}
		int32_t lowest = kLabelInf;
		while (__any(x > 0 && at < end)) {
			const bool go = x > 0 && at < end;
			const uint32_t a = at + sub;
			const bool own = go && a < end;
			int2 ends = make_int2(0, 0), p = make_int2(0, 0);
			int32_t l = kLabelInf;
			if (own) {
				ends = g.ends[a];
				p = g.pair[a];
				l = g.h[ends.x];
			}
			const bool open = own && p.x > threshold;
			const bool admissible = open && l == hv - 1;
			// the group's admissible residuals in arc order share the excess: running sums held at x
			const uint32_t cap = admissible ? (uint32_t)(p.x < x ? p.x : x) : 0u;
			uint32_t run = cap;
#pragma unroll
			for (int off = 1; off < kGroup; off <<= 1) {
				const uint32_t o = (uint32_t)__shfl_up((int)run, off, kGroup);
				const uint32_t s = run + o;
				run = sub >= off ? (s < (uint32_t)x ? s : (uint32_t)x) : run;
			}
			uint32_t before = (uint32_t)__shfl_up((int)run, 1, kGroup);
			before = sub == 0 ? 0u : before;
			const uint32_t room = (uint32_t)x - before;
			const int32_t f = (int32_t)(cap < room ? cap : room);
			const int32_t total = __shfl((int)run, kGroup - 1, kGroup);
			bool woken = false;
			if (f > 0) {
				g.pair[a] = make_int2(p.x - f, p.y + f);
				g.pair[ends.y] = make_int2(p.y + f, p.x - f);
				woken = atomicAdd(&g.e[ends.x], f) == 0;
			}
			stage_append(sh.next, woken, ends.x, out);
			if (own && ((open && !admissible) || (l > hv && p.y > threshold))) {
				lowest = l < lowest ? l : lowest;
			}
			x -= total;
			at += go ? (uint32_t)kGroup : 0u;
		}
#pragma unroll
		for (int off = kGroup / 2; off > 0; off >>= 1) {
			const int32_t o = __shfl_xor(lowest, off, kGroup);
			lowest = o < lowest ? o : lowest;
		}
		bool again = false;
		if (v >= 0 && sub == 0 && x0 > 0) {
			const int32_t sent = x0 - x;
			const int32_t left = sent > 0 ? atomicSub(&g.e[v], sent) - sent : x0;
			int32_t label = hv;
			if (x > 0) {
				const int32_t raised = lowest < kLabelInf ? lowest + 1 : kLabelInf;
				if (raised > hv) {
					g.h[v] = label = raised;
				}
			}
			again = left > 0 && label < kLabelInf;
		}
		stage_append(sh.next, again, v, out);
	}
}

// What workgroup 0 left in the control block before the last barrier.
__device__ inline int32_t told(const int32_t *word)
{
	return __hip_atomic_load(word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// A breadth-first search from its seeds. Returns the number of levels; a relabel's queue
// ends go to starts[1 ..], its active list to list[0] with its length in active_count.
template <int kGroup, bool kClosure>
__device__ inline int search(const CsrArgs &g, CsrShared &sh, CsrPhase &ph, int32_t threshold, int parity,
                             int32_t &active_count)
{
	const bool alone = gridDim.x == 1;
	const bool writer = blockIdx.x == 0 && threadIdx.x == 0;
	int32_t *counter = &g.ctl->active[parity];
	const CsrList active{g.list[0], nullptr, counter, alone};
	CsrList queue = step_list(g, ph, g.queue);
	search_seed<kClosure>(g, sh, ph, threshold, queue, active);
	int32_t got = step_end(g, sh, ph, queue);
	int level = 1, qs = 0, qe = got;
	if (!kClosure && writer) {
		g.starts[1] = qe;
		// the other round's count: every workgroup has read it before the barrier just passed
		__hip_atomic_store(&g.ctl->active[parity ^ 1], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
	}
	while (got > 0) {
		const bool handover = !alone && got <= g.solo_limit;
		if (handover) {
			// workgroup 0 runs the levels that follow while they stay short; the others wait for it
			if (blockIdx.x == 0) {
				ph.solo = true;
			}
		}
		if (!handover || blockIdx.x == 0) {
			do {
				queue = step_list(g, ph, g.queue + qe);
				search_level<kGroup, kClosure>(g, sh, ph, qs, qe, level, threshold, queue, active);
				got = step_end(g, sh, ph, queue);
				qs = qe;
				qe += got;
				++level;
				if (!kClosure && writer && got > 0) {
					g.starts[level] = qe;
				}
			} while (handover && got > 0 && got <= 4 * g.solo_limit);
		}
		if (handover) {
			ph.solo = false;
			if (writer) {
				g.ctl->solo[0] = level;
				g.ctl->solo[1] = qs;
				g.ctl->solo[2] = qe;
			}
			grid_phase_end(g, sh, ph);
			level = told(&g.ctl->solo[0]);
			qs = told(&g.ctl->solo[1]);
			qe = told(&g.ctl->solo[2]);
			got = qe - qs;
		}
	}
	if (!kClosure) {
		active_count = stage_flush(sh.active, active);
		if (alone) {
			__syncthreads();
		} else {
			grid_phase_end(g, sh, ph);
			active_count = told(counter);
		}
	}
	return level - 1;
}

// The stages of g.stages. The control block's barrier words, arrival count and gate must be zero, the
// rest as the last launch of the solve left it.
template <int kGroup>
__global__ __launch_bounds__(kCsrThreads) void k_csr_solve(CsrArgs g)
{
	__shared__ CsrShared sh;
	if (threadIdx.x == 0) {
		sh.next.count = 0;
		sh.active.count = 0;
	}
	__syncthreads();
	const bool alone = gridDim.x == 1;
	if (!alone && !all_running(g, sh)) {
		return;
	}
	const bool writer = blockIdx.x == 0 && threadIdx.x == 0;
	CsrPhase ph{0u, alone};
	int32_t threshold = g.ctl->threshold, rounds = g.ctl->rounds, count = g.ctl->list_count, levels = g.ctl->levels;
	int32_t status = g.ctl->status;
	long long sink = 0, passes = 0, steps = 0, cut_passes = 0;
	for (;;) {
		if (g.stages & kCsrRelabel) {
			if (rounds >= g.max_rounds) {
				status = kCsrNotConverged;
				break;
			}
			levels = search<kGroup, false>(g, sh, ph, threshold, rounds & 1, count);
			++rounds;
			passes += levels;
			if (count == 0) {
				if (threshold == 0) {
					status = kCsrDone;
					break;
				}
				threshold = 0;  // exact finish
			}
		}
		if (g.stages & kCsrPush) {
			const int limit = levels > kCsrMinSteps / 2 ? 2 * levels : kCsrMinSteps;
			int i = 0;
			while (i < limit && count > 0) {
				const bool handover = !alone && count <= g.solo_limit;
				if (handover && blockIdx.x == 0) {
					ph.solo = true;
				}
				if (!handover || blockIdx.x == 0) {
					do {
						const CsrList out = step_list(g, ph, g.list[(i & 1) ^ 1]);
						push_step<kGroup>(g, sh, ph, g.list[i & 1], count, out, threshold, sink);
						count = step_end(g, sh, ph, out);
						++i;
					} while (handover && i < limit && count > 0 && count <= 4 * g.solo_limit);
				}
				if (handover) {
					ph.solo = false;
					if (writer) {
						g.ctl->solo[0] = i;
						g.ctl->solo[1] = count;
					}
					grid_phase_end(g, sh, ph);
					i = told(&g.ctl->solo[0]);
					count = told(&g.ctl->solo[1]);
				}
			}
			steps += i;
		}
		if (!(g.stages & kCsrLoop)) {
			break;
		}
	}
	if ((g.stages & kCsrClosure) && status == kCsrDone) {
		int32_t unused;
		cut_passes = search<kGroup, true>(g, sh, ph, 0, 0, unused);
	}
	__syncthreads();
	const long long total = block_sum_i64<kCsrThreads>(sink, sh.red);
	if (threadIdx.x == 0 && total) {
		atomicAdd(&g.ctl->flow, (unsigned long long)total);
	}
	if (writer) {
		g.ctl->threshold = threshold;
		g.ctl->rounds = rounds;
		g.ctl->list_count = count;
		g.ctl->levels = levels;
		g.ctl->status = status;
		g.ctl->bfs_passes += passes;
		g.ctl->push_steps += steps;
		g.ctl->cut_passes = cut_passes;
	}
}

// Start of a solve: residuals, excess and residual sink links from the capacities.
__global__ __launch_bounds__(256) void k_csr_init(int n, int64_t arcs, const int32_t *__restrict__ cs,
                                                  const int32_t *__restrict__ ct, const int2 *__restrict__ cap,
                                                  int32_t *__restrict__ e, int32_t *__restrict__ rt,
                                                  int2 *__restrict__ pair, CsrControl *ctl, int32_t threshold)
{
	const int64_t start = (int64_t)blockIdx.x * blockDim.x + threadIdx.x, stride = (int64_t)gridDim.x * blockDim.x;
	for (int64_t v = start; v < n; v += stride) {
		e[v] = cs[v];
		rt[v] = ct[v];
	}
	for (int64_t a = start; a < arcs; a += stride) {
		pair[a] = cap[a];
	}
	if (start == 0) {
		*ctl = CsrControl{};
		ctl->threshold = threshold;
	}
}

// Before a further launch of a running solve: its barrier words and gate start at zero.
__global__ void k_csr_clear_words(CsrControl *ctl)
{
	if (threadIdx.x < 3) {
		ctl->word[threadIdx.x] = 0;
	}
	if (threadIdx.x == 0) {
		ctl->arrived = 0;
		ctl->gate = 0;
	}
}

}  // namespace cgp
