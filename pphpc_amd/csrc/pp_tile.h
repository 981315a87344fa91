/*
 * pp_tile.h -- the tile step: one kernel per iteration.
 *
 * The grid of every replica is cut into tiles of cells, one work-group each.
 * Between iterations a tile's agents lie in its own slot of a record buffer,
 * in id order (cells ascending, within a cell in acting order): they are the
 * state itself, an agent's id being the number of agents before it in the
 * replica, row by row. In one iteration a tile's group
 *   1. reads its own agents and those of the rows (and, where a grid row is
 *      cut into several tiles, the edge cells) next to it, moves each (one
 *      Philox block per agent: neighbours' agents on the border are moved by
 *      both tiles, which costs less than exchanging them would) and keeps
 *      those that land in the tile;
 *   2. sorts them by cell in LDS (a counting sort; agents of one cell are put
 *      in id order when the cell acts);
 *   3. acts on every occupied cell, the tile's grass being in LDS;
 *   4. writes the survivors and newborns, in order, to the other record
 *      buffer, with their number per tile, from which the next iteration
 *      derives the ids.
 * It replaces the three kernels of the staged step (sort, act, emit): one
 * launch, and each agent is read once and written once. Agents move one cell
 * along a row or a column (move_agent, pp_gpu.cl:744-821), so a tile reads no
 * more than its four neighbours' border cells.
 *
 * What bounds it: on small grids the chain of one group's phases (two round
 * trips to memory, eight barriers, and fetching some 20 KB of instructions
 * that each wave runs through about once); on large ones the vector units.
 * Per iteration, against the three staged kernels: 100 x 100 24.5 -> 6.8 us,
 * 400 x 400 27.5 -> 9.5, 1600 x 1600 41 -> 17.2, 12800 x 12800 768 -> 540;
 * 30 replicas of 1600 x 1600 402 -> 240.
 *
 * A tile that outgrows its LDS or border lists sets Ctl::stop; the tick
 * after it is then not run (every group of a later launch returns), and the
 * host goes on with smaller tiles or the staged step. Where the agents of all
 * replicas are more than the capacity, the batch fails with that tick, no tick
 * runs after it, and the records that it started from stay.
 *
 * Included by pp_sim.hip, inside its namespace.
 */

/* Where a replica's tiles are: tiles of bx x by cells, nbx to a grid row,
 * nby rows of them, tile0 the first; nbx == 1: bx = the grid's width. Cell
 * (x, r) of a tile has LDS cell index r * pitch + x. */
struct TileRep {
	uint32_t tile0, ntiles, nbx, nby, bx, by, shift, band0;
	/* its constants (Rep), here so that they come with one load */
	uint32_t slot, gx, gy, cb, t0, iters, cap, R;
	uint32_t key0, key1, sheep_gain, wolves_gain, sheep_thr, wolves_thr;
	uint32_t sheep_prob, wolves_prob, gxm, gxs;
};
/* ... in the constant address space: scalar loads, placed where they are used */
typedef __attribute__((address_space(4))) const TileRep TileRepC;

__device__ __forceinline__ TileRep tile_rep(const TileRep *p, uint32_t k) {
	const TileRepC *c = (const TileRepC *)p + k;
	TileRep r;
	r.tile0 = c->tile0; r.ntiles = c->ntiles; r.nbx = c->nbx; r.nby = c->nby;
	r.bx = c->bx; r.by = c->by; r.shift = c->shift; r.band0 = c->band0;
	r.slot = c->slot; r.gx = c->gx; r.gy = c->gy; r.cb = c->cb;
	r.t0 = c->t0; r.iters = c->iters; r.cap = c->cap; r.R = c->R;
	r.key0 = c->key0; r.key1 = c->key1;
	r.sheep_gain = c->sheep_gain; r.wolves_gain = c->wolves_gain;
	r.sheep_thr = c->sheep_thr; r.wolves_thr = c->wolves_thr;
	r.sheep_prob = c->sheep_prob; r.wolves_prob = c->wolves_prob;
	r.gxm = c->gxm; r.gxs = c->gxs;
	return r;
}

/* Sums of one tile's iteration, for the statistics row: sheep, wolves, grass
 * eaten, occupied cells, births, agents alive after the move, sheep energy,
 * wolf energy. */
struct TileStat {
	unsigned long long v[8];
};

/* Arguments of the tile kernels. A tile's header: its records, those in its
 * first and last row (low, high half), those in its edge lists (left, right),
 * and where its records start. They start in the tile's slot, or, when they
 * are more than it holds, in the spare records after the slots, taken with an
 * atomic add: these hold as many as there may be agents at all, so that they
 * run out only where the capacity is exceeded, too. */
struct TileArgs {
	const uint2 *in;       /* records: (x | r << 16, energy | V_WOLF) */
	uint2 *out;
	const uint4 *hin;
	uint4 *hout;
	const uint32_t *rin;   /* D2: per tile, the first record of each row */
	uint32_t *rout;
	uint32_t *idoff;       /* D2: per tile and row, id minus record index */
	uint32_t *rtot;        /* D2: agents per replica of the table */
	uint32_t *bsum;        /* D2: agents per band (row of tiles), two parities */
	const TileRep *trep;
	TileRep one;           /* the tiles of a table of one replica */
	const uint32_t *tk;    /* table entry of each tile */
	const uint32_t *bk;    /* table entry of each band */
	const TileStat *sin;
	TileStat *sout;
	TileStat *bstat;       /* D2: per band */
	unsigned long long *tot; /* outputs of a tick, three turns of PART_SLOTS */
	const uint2 *ein;      /* D2: edge lists, per tile left and right */
	uint2 *eout;
	uint32_t *spare;       /* spare records taken, by parity */
	uint32_t slot;         /* records of a slot */
	uint32_t spare0;       /* first spare record */
	uint32_t ntiles, nbands, nfin, par, rows;
	uint32_t nmax, hmax;   /* a tile's agents; a border row's */
};

constexpr uint32_t TILE_ROWS = 64;    /* rows of a tile, D2 */
constexpr uint32_t TILE_ECAP = 48;    /* records of an edge list */
constexpr uint32_t TILE_RESTAMP = 32; /* ticks between re-stamps of the grass */

/* The buffers (parity) that the last tick wrote: those whose tick is the
 * later. */
__device__ __forceinline__ uint32_t tile_last(const Ctl *ctl) {
	return (int32_t)(ctl->tt[1] - ctl->tt[0]) > 0 ? 1u : 0u;
}

/* The buffers that hold the state of Ctl::tick: those written last, or, when
 * the tick that wrote them failed the batch, those it started from (of which
 * the launch behind it may have counted on two ticks already). */
__host__ __device__ __forceinline__ uint32_t tile_cur(const Ctl *ctl) {
	return (ctl->tt[1] ^ ctl->tick) & 1u ? 0u : 1u;
}

/* Whether tick t may run: no error, and not at or past a stop. A stop set
 * during tick t names tick t + 1 (as t + 2: 0 is none), so it does not touch
 * the groups of tick t that start later; the first launch that does not run
 * halts the others, which would find the tick before in their buffers. */
__device__ __forceinline__ bool tile_runs(uint32_t error, uint32_t stop,
	uint32_t halt, uint32_t t) {
	return (error == 0) & (halt == 0) & ((stop == 0) | ((int32_t)(t + 1 - stop) < 0));
}

/* Sums of n statistics by a work-group, a lane to each counter: s_f[w][q] is
 * wave w's sum of counter q, complete after the barrier inside. */
template <int NT>
__device__ __forceinline__ void stat_sums(const TileStat *units, uint32_t n,
	unsigned long long (*s_f)[8]) {
	const uint32_t tid = threadIdx.x, q = tid & 7u;
	unsigned long long v = 0;
#pragma unroll 4
	for (uint32_t i = tid / 8; i < n; i += NT / 8) v += units[i].v[q];
#pragma unroll
	for (int o = 8; o < WAVE; o *= 2) v += __shfl_xor(v, o);
	if ((tid & (WAVE - 1)) < 8) s_f[tid / WAVE][q] = v;
	__syncthreads();
}

/* End of tick t for the k-th replica of the table, by one work-group: sums
 * the units' statistics (tiles, or bands of tiles), then does what
 * end_tick_solo and k_act_scan do. Nothing happens when the replica has
 * ended that tick already. Where the outputs of all replicas are more than
 * the capacity, the batch fails: the tick does not count, and no replica ends
 * it. */
template <int NT>
__device__ void tile_finish(const TileStat *units, uint32_t nunits, uint32_t k,
	uint32_t t, unsigned long long *tot, Ctl *ctl, const Tables &T,
	const Params &P, uint32_t nrep) {
	__shared__ unsigned long long s_f[NT / WAVE][8];
	const uint32_t tid = threadIdx.x, lane = tid & (WAVE - 1), w = tid / WAVE;
	const uint32_t slot = nrep == 1 ? P.one_slot : T.order[k];
	RepCtl &rc = T.rctl[slot];
	const Rep &rp = T.rep[slot];
	const uint32_t s = t - rp.t0;
	const bool failed = ctl->error != 0;
	const bool due = rc.status == RS_ACTIVE && rc.step == s && !failed;
	stat_sums<NT>(units, due ? nunits : 0u, s_f);
	if (w != 0) return;
	/* the outputs of all replicas, which the agent buffers bound */
	unsigned long long total = 0;
	if (nrep > 1) total = wave_sum(tot[(t % 3) * PART_SLOTS + lane]);
	unsigned long long sum = 0, a[8];
	if (lane < 8)
#pragma unroll 1
		for (int q = 0; q < NT / WAVE; q++) sum += s_f[q][lane];
#pragma unroll
	for (int i = 0; i < 8; i++) a[i] = __shfl(sum, i);
	if (lane != 0) return;
	/* (the tick counts on when every replica is done; one replica's total:
	 * below) */
	if (k == 0 && !failed && total <= P.cap && (int32_t)(t + 1 - ctl->tick) > 0)
		ctl->tick = t + 1;
	if (!due) return;
	const unsigned long long out64 = a[0] + a[1];
	if (nrep == 1) total = out64;
	if (total > P.cap) {
		if (k == 0) ctl->tick = t;
		set_error(ctl, PP_OUT_OF_RESOURCES, t, -1);
		return;
	}
	const uint32_t out = (uint32_t)out64;
	atomicAdd(&ctl->sum_live, a[5]);
	atomicAdd(&ctl->sum_out, out64);
	const bool over = rc.ovf == t + 1;
	if (over || out > rp.cap) {
		rc.status = RS_FAILED;
		rc.error = over ? PP_ENERGY_OVERFLOW : PP_OUT_OF_RESOURCES;
		rc.err_step = s;
		rc.n = 0;
		return;
	}
	const uint32_t M = rp.R + 1;
	unsigned long long D = rc.dead_cells, S = rc.cd_sum;
	S -= D;
	const uint32_t expire = (t + 1) % M;
	D -= rp.ring[expire];
	rp.ring[expire] = 0;
	const unsigned long long E = a[2];
	rp.ring[t % M] += E;
	D += E;
	S += E * (unsigned long long)rp.R;
	rc.dead_cells = D;
	rc.cd_sum = S;
	pp_stats64_t *row = &rp.stats[(s + 1) % rp.stats_rows];
	row->sheep = a[0];
	row->wolves = a[1];
	row->grass = (unsigned long long)rp.C - D;
	row->sheep_en = a[6];
	row->wolves_en = a[7];
	row->grass_en = S;
	row->errors = 0;
	atomicAdd(&ctl->agent_steps, (unsigned long long)rc.n);
	atomicAdd(&ctl->sum_occ, a[3]);
	atomicAdd(&ctl->sum_eaten, E);
	atomicAdd(&ctl->sum_births, a[4]);
	rc.agent_steps += rc.n;
	rc.step = s + 1;
	rc.n = out;
	if (s + 1 >= rp.iters) {
		rc.status = RS_DONE;
		rc.n = 0;
	}
}

/* One cell of k agents (2 <= k <= N <= 8) at LDS slots p .. p + k - 1, in
 * registers: the steps of k_act's register path, the starting order being
 * the agents' id order (their ranks) instead of the slots'. Written without
 * branches (places from k on hold no agent): a wave runs through it about
 * once, so its length is what it costs. The acted values go back to the slots
 * in acting order. Returns whether the grass was eaten; *ovf is set by an
 * agent above the energy limit. (Slots up to p + N - 1 are read.) */
template <uint32_t N>
__device__ __forceinline__ bool tile_cell(uint32_t *s_val, const uint32_t *s_id,
	uint32_t p, uint32_t k, bool grass, uint32_t c_local, uint32_t step,
	uint32_t key0, uint32_t key1, uint32_t sheep_gain, uint32_t wolves_gain,
	uint32_t sheep_thr, uint32_t wolves_thr, uint32_t *ovf) {
	static_assert(N == 4 || N == 8, "4-bit indices in one word");
	uint32_t id[N], v0[4];
#pragma unroll
	for (uint32_t q = 0; q < N; q++) id[q] = lds_ld(s_id + p + q);
	if constexpr (N == 4)
#pragma unroll
		for (uint32_t q = 0; q < 4; q++) v0[q] = lds_ld(s_val + p + q);
	const uint4 w0 = pp_philox(c_local, step, PP_STREAM_SHUFFLE, 0, key0, key1);
	uint4 w1 = make_uint4(0, 0, 0, 0);
	if constexpr (N == 8)
		w1 = pp_philox(c_local, step, PP_STREAM_SHUFFLE, 1, key0, key1);
#pragma unroll
	for (uint32_t q = 0; q < N; q++) id[q] = q < k ? id[q] : 0xFFFFFFFFu;
	/* ranks by id: of each pair one comes first */
	uint32_t rank[N];
#pragma unroll
	for (uint32_t q = 0; q < N; q++) rank[q] = 0;
#pragma unroll
	for (uint32_t q = 0; q < N; q++)
#pragma unroll
		for (uint32_t o = q + 1; o < N; o++) {
			const uint32_t lt = id[q] < id[o] ? 1u : 0u;
			rank[o] += lt;
			rank[q] += 1u - lt;
		}
	uint32_t perm = 0;
#pragma unroll
	for (uint32_t q = 0; q < N; q++) perm |= q << (4 * rank[q]);
	/* Fisher-Yates from place k - 1 down, draw m = k - 1 - i for place i */
#pragma unroll
	for (uint32_t i = N - 1; i >= 1; i--) {
		const uint32_t m = k - 1 - i;
		uint32_t word = m == 0 ? w0.x : m == 1 ? w0.y : m == 2 ? w0.z : w0.w;
		if constexpr (N == 8) {
			const uint32_t hi = m == 4 ? w1.x : m == 5 ? w1.y : w1.z;
			word = m >= 4 ? hi : word;
		}
		const uint32_t jj = i < k ? pp_bounded(word, i + 1) : i;
		const uint32_t x = ((perm >> (4 * i)) ^ (perm >> (4 * jj))) & 0xFu;
		perm ^= (x << (4 * i)) | (x << (4 * jj));
	}
	uint32_t V[N];
	uint32_t sheep = 0;
	const uint32_t there = (1u << k) - 1u;
#pragma unroll
	for (uint32_t q = 0; q < N; q++) {
		const uint32_t at = (perm >> (4 * q)) & 0xFu;
		if constexpr (N == 4) {
			const uint32_t a = (at & 1u) ? v0[1] : v0[0], b = (at & 1u) ? v0[3] : v0[2];
			V[q] = (at & 2u) ? b : a;
		} else {
			V[q] = lds_ld(s_val + p + at);
		}
		sheep |= (V[q] & V_WOLF) ? 0u : 1u << q;
	}
	sheep &= there;
	uint32_t killed = 0, g = grass ? 1u : 0u, over = 0;
#pragma unroll
	for (uint32_t q = 0; q < N; q++) {
		const uint32_t v = V[q];
		const bool acts = ((there & ~killed) >> q) & 1u, wolf = (v & V_WOLF) != 0;
		const uint32_t prey = sheep & ~killed;
		const uint32_t hunt = acts & wolf ? prey & (0u - prey) : 0u;
		const uint32_t graze = acts & !wolf ? g : 0u;
		killed |= hunt;
		g ^= graze;
		int32_t e = (int32_t)(v & V_ENERGY);
		e += (int32_t)((hunt ? wolves_gain : 0u) + (graze ? sheep_gain : 0u));
		const bool child = acts & (e > (int32_t)(wolf ? wolves_thr : sheep_thr)) &
			((v & V_REPRO) != 0);
		const uint32_t flags = V_CHILD | ((e & 1) ? V_ODD : 0u);
		e -= child ? e >> 1 : 0;
		over |= e > (int32_t)V_ENERGY ? 1u : 0u;
		V[q] = (v & V_WOLF) | (child ? flags : 0u) | ((uint32_t)e & V_ENERGY);
	}
#pragma unroll
	for (uint32_t q = 0; q < N; q++)
		if (q < k) lds_st(s_val + p + q, V[q] | (((killed >> q) & 1u) ? V_KILLED : 0u));
	*ovf |= over;
	return grass && !g;
}

/* The same for a cell of any number of agents, in LDS. */
__device__ __forceinline__ bool tile_cell_any(uint32_t *s_val_, uint32_t *s_id_,
	uint32_t p, uint32_t k, bool grass, uint32_t c_local, uint32_t step,
	uint32_t key0, uint32_t key1, uint32_t sheep_gain, uint32_t wolves_gain,
	uint32_t sheep_thr, uint32_t wolves_thr, uint32_t *ovf) {
	uint32_t *s_val = s_val_ + p, *s_id = s_id_ + p;
	for (uint32_t i = 1; i < k; i++) {
		const uint32_t id = lds_ld(s_id + i), v = lds_ld(s_val + i);
		uint32_t j = i;
		while (j > 0 && lds_ld(s_id + j - 1) > id) {
			lds_st(s_id + j, lds_ld(s_id + j - 1));
			lds_st(s_val + j, lds_ld(s_val + j - 1));
			j--;
		}
		lds_st(s_id + j, id);
		lds_st(s_val + j, v);
	}
	uint4 r = make_uint4(0, 0, 0, 0);
	for (uint32_t i = k - 1, m = 0; i > 0; i--, m++) {
		if ((m & 3u) == 0)
			r = pp_philox(c_local, step, PP_STREAM_SHUFFLE, m >> 2, key0, key1);
		const uint32_t word = (m & 3u) == 0 ? r.x : (m & 3u) == 1 ? r.y
			: (m & 3u) == 2 ? r.z : r.w;
		const uint32_t jj = pp_bounded(word, i + 1);
		if (jj != i) {
			const uint32_t a = lds_ld(s_val + i);
			lds_st(s_val + i, lds_ld(s_val + jj));
			lds_st(s_val + jj, a);
		}
	}
	bool ate = false;
	for (uint32_t q = 0; q < k; q++) {
		const uint32_t v = lds_ld(s_val + q);
		if (v & V_KILLED) continue;
		int32_t e = (int32_t)(v & V_ENERGY);
		uint32_t thr;
		if (!(v & V_WOLF)) {
			if (grass) {
				grass = false;
				ate = true;
				e += (int32_t)sheep_gain;
			}
			thr = sheep_thr;
		} else {
			for (uint32_t o = 0; o < k; o++) {
				const uint32_t u = lds_ld(s_val + o);
				if (!(u & (V_WOLF | V_KILLED))) {
					lds_st(s_val + o, u | V_KILLED);
					e += (int32_t)wolves_gain;
					break;
				}
			}
			thr = wolves_thr;
		}
		uint32_t nv = v & V_WOLF;
		if (e > (int32_t)thr && (v & V_REPRO)) {
			nv |= V_CHILD | ((e & 1) ? V_ODD : 0u);
			e -= e / 2;
		}
		if (e > (int32_t)V_ENERGY) *ovf = 1;
		lds_st(s_val + q, nv | ((uint32_t)e & V_ENERGY));
	}
	return ate;
}

/* Geometry of one tile. */
struct TileGeo {
	uint32_t x0, y0, w, h;       /* its cells */
	uint32_t up, down, left, right;
	uint32_t pitch;
};

template <bool D2>
__device__ __forceinline__ TileGeo tile_geo(const TileRep &tr, uint32_t lt,
	uint32_t gx, uint32_t gy) {
	TileGeo g;
	const uint32_t ty = D2 ? lt / tr.nbx : lt, tx = D2 ? lt - ty * tr.nbx : 0u;
	g.x0 = tx * tr.bx;
	g.y0 = ty * tr.by;
	g.w = min(tr.bx, gx - g.x0);
	g.h = min(tr.by, gy - g.y0);
	const uint32_t yu = ty ? ty - 1 : tr.nby - 1, yd = ty + 1 < tr.nby ? ty + 1 : 0;
	if (D2) {
		const uint32_t xl = tx ? tx - 1 : tr.nbx - 1, xr = tx + 1 < tr.nbx ? tx + 1 : 0;
		g.up = tr.tile0 + yu * tr.nbx + tx;
		g.down = tr.tile0 + yd * tr.nbx + tx;
		g.left = tr.tile0 + ty * tr.nbx + xl;
		g.right = tr.tile0 + ty * tr.nbx + xr;
		g.pitch = 1u << tr.shift;
	} else {
		g.up = tr.tile0 + yu;
		g.down = tr.tile0 + yd;
		g.left = g.right = 0;
		g.pitch = gx;
	}
	return g;
}

/* 16 bytes of grass at any address (the hardware takes unaligned vectors). */
struct __attribute__((packed, aligned(1))) Grass16 {
	uint32_t v[4];
};

/* The tile's grass as rows of 16-byte chunks: one row of w * h cells (D2
 * false: the tile's cells are contiguous), or h rows of w cells, 2^csh chunks
 * apart in LDS. A cell's place in LDS is its cell index. Rows start at any
 * address: loading and storing 32-bit words at multiples of four, with each
 * row's first cell anywhere in its first word, was a quarter of the kernel's
 * instructions where rows are not whole chunks (4001 x 2999: 55 -> 49 us an
 * iteration, 48 replicas of mixed sizes 102 -> 92, 1013 x 487 11.4 -> 10.8). */
template <typename GT, bool D2>
struct TileGrass {
	static constexpr uint32_t VPC = 16 / sizeof(GT);   /* cells of a chunk */
	uint32_t start, gx, n, csh, rows;
	__device__ __forceinline__ TileGrass(uint32_t cell0, uint32_t gx_, uint32_t w,
		uint32_t h, uint32_t shift) {
		start = cell0;
		gx = gx_;
		n = D2 ? w : w * h;
		rows = h;
		csh = shift - (VPC == 16 ? 4u : VPC == 8 ? 3u : 2u);
	}
	/* chunk i (in LDS order): its first cell and how many of its cells the
	 * tile has; false: none */
	__device__ __forceinline__ bool chunk(uint32_t i, uint32_t &cell,
		uint32_t &cells) const {
		uint32_t r = 0, x = i * VPC;
		if (D2) {
			r = i >> csh;
			x = (i & ((1u << csh) - 1)) * VPC;
		}
		cell = start + r * gx + x;
		cells = n - x;
		return x < n && (!D2 || r < rows);
	}
};

/* One iteration of every tile (see the head of this file). Blocks
 * [0, nfin) end the tick before for a replica each, beside the others. */
template <typename GT, int NT, int IPT, uint32_t CELLS, bool D2, bool SOLO>
__global__ __launch_bounds__(NT) void k_tile(TileArgs A, Ctl *ctl, Tables T,
	Params P, uint32_t nrep, GT *grass) {
	constexpr uint32_t AG = NT * IPT, NW = NT / WAVE;
	constexpr uint32_t WPT = CELLS / 2 / NT;   /* counter words a thread scans */
	using TG = TileGrass<GT, D2>;
	constexpr uint32_t CHUNKS = CELLS / TG::VPC, VIT = (CHUNKS + NT - 1) / NT;
	constexpr uint32_t NWT = NW * IPT > WAVE ? 2u : 1u;   /* waves' counts a lane scans */
	static_assert(AG < 65536 && CELLS < 65536, "16-bit slots and cells");
	static_assert(NW * IPT <= 2 * WAVE, "one wave scans the waves' counts");
	static_assert(WPT * NT * 2 == CELLS && WPT % 2 == 0, "counter words");
	__shared__ __align__(16) uint32_t s_cnt[CELLS / 2 + 4];
	__shared__ uint32_t s_val[AG + 8];
	__shared__ uint32_t s_id[AG + 8];
	__shared__ uint16_t s_cell[AG + 2];
	__shared__ uint16_t s_list[AG / 2];   /* first slots of cells with several agents */
	__shared__ uint32_t s_row[D2 ? TILE_ROWS + 1 : 2];   /* first slots of rows */
	__shared__ uint4 s_grass[CHUNKS];
	__shared__ uint32_t s_tmp[NW], s_sum[2 * NW], s_wt[NWT * WAVE];
	__shared__ uint32_t s_idoff[D2 ? 3 * TILE_ROWS : 1];
	__shared__ unsigned long long s_red[NW][8];   /* in TileStat's order */
	__shared__ uint32_t s_nlist, s_ovf, s_go, s_edge[2];

	const uint32_t tid = threadIdx.x, lane = tid & (WAVE - 1);
	const uint32_t w = __builtin_amdgcn_readfirstlane(tid / WAVE);
	/* A group that has its CU to itself waits for each of its first loads, and
	 * a scalar load is waited for together with every other one, so that a
	 * chain of six round trips stood before the first barrier (1.5 us): all
	 * arguments that they need are taken at once, and the uniform values come
	 * as vector loads, a word a lane (100 x 100: 7.9 -> 7.7 us). In tiles of
	 * 256 columns, where other groups fill the wait, scalar loads are the
	 * faster (12800 x 12800: 577 us, 620 with vector loads, which queue behind
	 * the records). */
	if (!D2)
		asm volatile("" :: "s"(A.in), "s"(A.hin), "s"(grass), "s"(ctl), "s"(T.rctl),
			"s"(A.slot), "s"(A.ntiles), "s"(A.nfin), "s"(A.par));
	if (SOLO && !D2)
		asm volatile("" :: "s"(A.one.tile0), "s"(A.one.ntiles), "s"(A.one.gx),
			"s"(A.one.gy), "s"(A.one.cb), "s"(A.one.slot), "s"(A.one.by), "s"(A.one.nby));
	uint32_t cw = 0;
	if (!D2) cw = reinterpret_cast<const uint32_t *>(ctl)[lane & 15u];
	static_assert(offsetof(Ctl, error) == 4 * 4 && offsetof(Ctl, tt) == 12 * 4 &&
		offsetof(Ctl, stop) == 14 * 4 && offsetof(Ctl, halt) == 15 * 4, "words of Ctl");
	auto ctl_word = [&](uint32_t i) {
		return D2 ? reinterpret_cast<const uint32_t *>(ctl)[i]
			: (uint32_t)__builtin_amdgcn_readlane((int)cw, (int)i);
	};
	if (blockIdx.x < A.nfin) {
		const uint32_t k = blockIdx.x, tick = ctl_word(12 + A.par);
		const bool runs = tile_runs(ctl_word(4), ctl_word(14), ctl_word(15), tick);
		if (k == 0) {
			if (tid == 0) {
				if (runs) {
					ctl->tt[1 - A.par] = tick + 1;
					A.spare[A.par] = 0;   /* for the next tick's outputs */
				} else {
					ctl->halt = 1;
				}
			}
			if (!SOLO && tid < PART_SLOTS)
				A.tot[((tick + 1) % 3) * PART_SLOTS + tid] = 0;
		}
		const TileRep tr = SOLO ? A.one : tile_rep(A.trep, k);
		if (D2) tile_finish<NT>(A.bstat + tr.band0, tr.nby, k, tick - 1, A.tot, ctl, T,
				P, nrep);
		else tile_finish<NT>(A.sin + tr.tile0, tr.ntiles, k, tick - 1, A.tot, ctl, T, P,
				nrep);
		return;
	}
	/* groups of one XCD take neighbouring tiles (their borders are then read
	 * through one L2) */
	const uint32_t b = blockIdx.x - A.nfin, per = (A.ntiles + NXCD - 1) / NXCD;
	const uint32_t tile = (b % NXCD) * per + b / NXCD;
	if (b / NXCD >= per || tile >= A.ntiles) return;
	const uint32_t k = SOLO ? 0u : __builtin_amdgcn_readfirstlane(A.tk[tile]);
	const TileRep tr = SOLO ? A.one : tile_rep(A.trep, k);
	const uint32_t gx = tr.gx, gy = tr.gy, cb = tr.cb;
	const uint32_t key0 = tr.key0, key1 = tr.key1;
	const uint32_t lt = tile - tr.tile0;
	const TileGeo g = tile_geo<D2>(tr, lt, gx, gy);
	const bool wrapx = tr.nbx == 1, wrapy = tr.nby == 1;
	/* headers: this tile's, up, down, left, right */
	uint4 hs[5];
	uint32_t hw = 0, rw = 0, d2_status = 0, d2_over = 0;
	if (D2) {
		hs[0] = A.hin[tile];
		hs[1] = A.hin[g.up];
		hs[2] = A.hin[g.down];
		hs[3] = A.hin[g.left];
		hs[4] = A.hin[g.right];
		d2_status = T.rctl[tr.slot].status;
		d2_over = T.rctl[tr.slot].ovf;
	} else {
		uint32_t ht = tile;
		if (lane >= 4) ht = g.up;
		if (lane >= 8) ht = g.down;
		hw = reinterpret_cast<const uint32_t *>(A.hin)[ht * 4 + (lane & 3u)];
		rw = reinterpret_cast<const uint32_t *>(T.rctl + tr.slot)[lane & 7u];
	}
	static_assert(offsetof(RepCtl, status) == 3 * 4 && offsetof(RepCtl, ovf) == 6 * 4,
		"words of RepCtl");
	auto header = [&](uint32_t i) {
		const uint4 h = hs[i >> 2];
		const uint32_t j = i & 3u;
		return D2 ? (j == 0 ? h.x : j == 1 ? h.y : j == 2 ? h.z : h.w)
			: (uint32_t)__builtin_amdgcn_readlane((int)hw, (int)i);
	};
	/* No replica moves when the outputs of the last tick are more than the
	 * capacity (the first groups then fail the batch): the records which that
	 * tick started from stay, as its outputs may not all have been written.
	 * (One replica: total_in, below; cut rows: k_tile_scan halts. Requested
	 * before the grass, which would be waited for with it.) */
	uint32_t outputs = 0;
	if (!SOLO && !D2 && w == 0)
		outputs = (uint32_t)A.tot[((ctl_word(12 + A.par) + 2) % 3) * PART_SLOTS + lane];
	/* the ids: the agents of the replica's tiles before this one */
	uint32_t bef = 0, all = 0;
	if (!D2) {
		if (tid < tr.ntiles) all = A.hin[tr.tile0 + tid].x;
	}
	if (D2 && tid < 3 * TILE_ROWS) {
		const uint32_t q = tid / TILE_ROWS, r = tid % TILE_ROWS;
		if (r < g.h) {
			const uint32_t tl = g.left, tg = g.right;
			uint32_t t = tile;
			if (q == 1) t = tl;
			if (q == 2) t = tg;
			s_idoff[tid] = A.idoff[t * A.rows + r];
		}
	}
	/* the grass, requested now and staged in LDS after the records are (a last
	 * chunk may run on into the next row or replica: those cells are not
	 * used) */
	const TG G(cb + g.y0 * gx + g.x0, gx, g.w, g.h, tr.shift);
	Grass16 gq[VIT];
#pragma unroll
	for (uint32_t i = 0; i < VIT; i++) {
		uint32_t cell, cells;
		gq[i] = Grass16{{0, 0, 0, 0}};
		if (G.chunk(i * NT + tid, cell, cells))
			gq[i] = *reinterpret_cast<const Grass16 *>(grass + cell);
	}
	for (uint32_t i = tid; i < CELLS / 8 + 1; i += NT)
		*reinterpret_cast<uint4 *>(s_cnt + 4 * i) = make_uint4(0, 0, 0, 0);
	if (tid < NWT * WAVE) s_wt[tid] = 0;
	const uint32_t tick = ctl_word(12 + A.par), step = tick - tr.t0;
	/* (words are taken from their lanes outside of branches, where all lanes
	 * have loaded) */
	const uint32_t status = D2 ? d2_status
		: (uint32_t)__builtin_amdgcn_readlane((int)rw, 3);
	const uint32_t over = D2 ? d2_over
		: (uint32_t)__builtin_amdgcn_readlane((int)rw, 6);
	/* A replica that is done or has failed no longer moves. Its status is
	 * that before or after the end of the last tick, written beside this:
	 * both give the same answer. (One thread decides for the group: an energy
	 * limit or an error may be noted meanwhile.) */
	const bool fits = SOLO || D2 || w != 0 || wave_sum32(outputs) <= P.cap;
	const bool go = tile_runs(ctl_word(4), ctl_word(14), ctl_word(15), tick) &
		fits & (status == RS_ACTIVE) & (step < tr.iters) &
		((over == 0) | (over == tick + 1));
	if (tid == 0) {
		s_nlist = 0;
		s_ovf = 0;
		s_edge[0] = s_edge[1] = 0;
		s_go = go;
	}
	uint32_t idb = 0, idb_up = 0, idb_dn = 0, total_in;
	if (!D2) {
		bef = tid < lt ? all : 0u;
		for (uint32_t i = tid + NT; i < tr.ntiles; i += NT) {
			const uint32_t n = A.hin[tr.tile0 + i].x;
			all += n;
			bef += i < lt ? n : 0u;
		}
		all = wave_sum32(all);
		bef = wave_sum32(bef);
		if (lane == 0) {
			s_sum[2 * w] = all;
			s_sum[2 * w + 1] = bef;
		}
	}
	__syncthreads();
	if (!D2) {
		uint32_t a = 0, c = 0;
#pragma unroll
		for (uint32_t i = 0; i < NW; i++) {
			a += s_sum[2 * i];
			c += s_sum[2 * i + 1];
		}
		total_in = __builtin_amdgcn_readfirstlane(a);
		idb = __builtin_amdgcn_readfirstlane(c);
	} else {
		total_in = __builtin_amdgcn_readfirstlane(A.rtot[k]);
	}
	if (!s_go || total_in > tr.cap || total_in > P.cap) return;

	const uint32_t n0 = header(0);
	const uint32_t nup = wrapy ? 0u : header(4 + 1) >> 16;
	const uint32_t ndn = wrapy ? 0u : header(8 + 1) & 0xFFFFu;
	const uint32_t nl = D2 && !wrapx ? header(12 + 2) >> 16 : 0u;
	const uint32_t nr = D2 && !wrapx ? header(16 + 2) & 0xFFFFu : 0u;
	const uint32_t i1 = n0, i2 = i1 + nup, i3 = i2 + ndn, i4 = i3 + nl, i5 = i4 + nr;
	if (i5 > AG) {
		/* (the limits set when the records were written exclude this) */
		if (tid == 0) set_error(ctl, PP_LIBRARY_ERROR, tick, (int32_t)tile);
		return;
	}
	/* positions and ids of the ranges, as offsets from the item index */
	const uint32_t first_up = header(4) - nup;
	const uint32_t p_own = header(3);
	const uint32_t p_up = header(4 + 3) + first_up - i1;
	const uint32_t p_dn = header(8 + 3) - i2;
	uint32_t p_l = 0, p_r = 0;
	if (!D2) {
		idb_up = (lt ? idb - header(4)
			: total_in - header(4)) + first_up - i1;
		idb_dn = (lt + 1 < tr.ntiles ? idb + n0 : 0u) - i2;
	} else {
		const uint32_t uh = min(tr.by, gy - (g.y0 ? g.y0 - tr.by : (tr.nby - 1) * tr.by));
		idb_up = __builtin_amdgcn_readfirstlane(A.idoff[g.up * A.rows + uh - 1])
			+ first_up - i1;
		idb_dn = __builtin_amdgcn_readfirstlane(A.idoff[g.down * A.rows]) - i2;
		/* the right list of the tile left of this one, and vice versa */
		p_l = (2 * g.left + 1) * TILE_ECAP - i3;
		p_r = 2 * g.right * TILE_ECAP - i4;
	}
	uint2 rec[IPT];
	uint32_t pk[IPT], vv[IPT], ids[IPT];
#pragma unroll
	for (int j = 0; j < IPT; j++) {
		rec[j] = make_uint2(0u, 0u);
		pk[j] = 0xFFFFFFFFu;
		vv[j] = ids[j] = 0;
	}
#pragma unroll
	for (int j = 0; j < IPT; j++) {
		if ((uint32_t)j * NT >= i5) break;   /* (uniform: no more rounds) */
		const uint32_t i = j * NT + tid;
		if ((uint32_t)(j + 1) * NT <= i1) {
			rec[j] = A.in[p_own + i];     /* a round of own agents */
		} else if (i < i5) {
			uint32_t p = i < i1 ? p_own : i < i2 ? p_up : p_dn;
			if (D2 && i >= i3) p = i < i4 ? p_l : p_r;
			const uint2 *src = D2 && i >= i3 ? A.ein : A.in;
			rec[j] = src[(uint32_t)(p + i)];
		}
	}
	/* grass to LDS: arrived before the records, in issue order */
#pragma unroll
	for (uint32_t i = 0; i < VIT; i++)
		if (VIT * NT == CHUNKS || i * NT + tid < CHUNKS)
			s_grass[i * NT + tid] = make_uint4(gq[i].v[0], gq[i].v[1], gq[i].v[2], gq[i].v[3]);

	/* 1. the moves; an agent that lands is counted in its cell and keeps its
	 * place among the cell's arrivals */
#pragma unroll
	for (int j = 0; j < IPT; j++) {
		if ((uint32_t)j * NT >= i5) break;
		const uint32_t i = j * NT + tid;
		if (i >= i5) continue;
		int32_t x = (int32_t)(rec[j].x & 0xFFFFu), r = (int32_t)(rec[j].x >> 16);
		uint32_t id = i + (D2 ? s_idoff[r] : idb);
		if ((uint32_t)(j + 1) * NT > i1) {
			/* a round with neighbours' agents */
			if (!D2) {
				id = i + (i < i1 ? idb : i < i2 ? idb_up : idb_dn);
				r = i < i1 ? r : i < i2 ? -1 : (int32_t)g.h;
			} else if (i >= i3) {
				/* an edge record's x is its index among its tile's records */
				id = (uint32_t)x + s_idoff[(i < i4 ? 1u : 2u) * TILE_ROWS + (uint32_t)r];
				x = i < i4 ? -1 : (int32_t)g.w;
			} else if (i >= i1) {
				id = i + (i < i2 ? idb_up : idb_dn);
				r = i < i2 ? -1 : (int32_t)g.h;
			}
		}
		const uint4 d4 = pp_philox(id, step, PP_STREAM_MOVE, 0, key0, key1);
		const uint32_t dice = pp_bounded(d4.y, 100);
		/* the direction's steps along x and y, from tables of 2-bit signed
		 * entries: 0, 1, -1, 0, 0 and 0, 0, 0, 1, -1 */
		const uint32_t dir2 = 2 * pp_bounded(d4.x, 5);
		x += __builtin_amdgcn_sbfe(0x34, dir2, 2);
		r += __builtin_amdgcn_sbfe(0x340, dir2, 2);
		if (wrapx) x = x < 0 ? (int32_t)g.w - 1 : x == (int32_t)g.w ? 0 : x;
		if (wrapy) r = r < 0 ? (int32_t)g.h - 1 : r == (int32_t)g.h ? 0 : r;
		/* it loses one energy, and dies below one */
		const uint32_t y = rec[j].y;
		if (((y & V_ENERGY) < 2) | ((uint32_t)x >= g.w) | ((uint32_t)r >= g.h)) continue;
		const uint32_t c = __umul24((uint32_t)r, g.pitch) + (uint32_t)x, sh = (c & 1u) * 16;
		const uint32_t old = atomicAdd(&s_cnt[c >> 1], 1u << sh);
		pk[j] = c | (((old >> sh) & 0xFFFFu) << 16);
		vv[j] = (y - 1) | (dice < ((y & V_WOLF) ? tr.wolves_prob : tr.sheep_prob) ?
			V_REPRO : 0u);
		ids[j] = id;
	}
	__syncthreads();

	/* 2. first slot of every cell, then the agents to their slots */
	uint32_t L;
	{
		uint32_t v[WPT];
		uint2 *p2 = reinterpret_cast<uint2 *>(s_cnt + WPT * tid);
#pragma unroll
		for (uint32_t i = 0; i < WPT / 2; i++) {
			const uint2 u = p2[i];
			v[2 * i] = u.x;
			v[2 * i + 1] = u.y;
		}
		uint32_t sum = 0;
#pragma unroll
		for (uint32_t i = 0; i < WPT; i++) sum += v[i];
		sum = (sum & 0xFFFFu) + (sum >> 16);
		const uint32_t x = wave_incl_scan32(sum);
		if (lane == WAVE - 1) s_tmp[w] = x;
		__syncthreads();
		uint32_t run = x - sum, tot = 0;
#pragma unroll
		for (uint32_t i = 0; i < NW; i++) {
			const uint32_t t = s_tmp[i];
			run += i < w ? t : 0u;
			tot += t;
		}
		L = __builtin_amdgcn_readfirstlane(tot);
#pragma unroll
		for (uint32_t i = 0; i < WPT / 2; i++) {
			uint32_t o[2];
#pragma unroll
			for (uint32_t q = 0; q < 2; q++) {
				const uint32_t lo = v[2 * i + q] & 0xFFFFu;
				o[q] = run | ((run + lo) << 16);
				run += lo + (v[2 * i + q] >> 16);
			}
			p2[i] = make_uint2(o[0], o[1]);
		}
		if (tid == 0) s_cnt[CELLS / 2] = L;
	}
	__syncthreads();
	const uint16_t *s_start = reinterpret_cast<const uint16_t *>(s_cnt);
#pragma unroll
	for (int j = 0; j < IPT; j++) {
		if ((uint32_t)j * NT >= i5) break;
		if (pk[j] == 0xFFFFFFFFu) continue;
		const uint32_t c = pk[j] & 0xFFFFu, c0 = s_start[c];
		const uint32_t q = c0 + (pk[j] >> 16);
		/* a cell with several agents is listed by the second that came (the
		 * asm keeps the compiler from first adding up lanes that share an
		 * atomic, which takes more than the few atomics do) */
		if (pk[j] >> 16 == 1) {
			uint32_t z = 0;
			asm("" : "+v"(z));
			s_list[atomicAdd(&s_nlist + z, 1u)] = (uint16_t)c0;
		}
		s_val[q] = vv[j];
		s_id[q] = ids[j];
		s_cell[q + 1] = (uint16_t)c;
	}
	/* first slot of each row (else: of the second and the last) */
	if (D2) {
		for (uint32_t r = tid; r < g.h; r += NT) s_row[r] = s_start[r * g.pitch];
	} else if (tid < 2) {
		s_row[tid] = s_start[(tid ? g.h - 1 : g.h > 1 ? 1u : 0u) * g.pitch];
	}
	if (tid == 0) {
		s_cell[0] = 0xFFFFu;
		s_cell[L + 1] = 0xFFFFu;
	}
	__syncthreads();

	/* 3. actions: the listed cells, dealt out from the last lane on, and
	 * those of one agent, from the first: where there are few of both,
	 * different waves act on them at the same time (100 x 100: 7.7 -> 7.3 us,
	 * 12800 x 12800 576 -> 561, against those of one agent first, listing the
	 * others, and these after a barrier; with a cell's single agent acting
	 * from its registers in the loop above 7.5 and 548, 1600 x 1600 18.4 ->
	 * 18.7) */
	const uint32_t sheep_gain = tr.sheep_gain, wolves_gain = tr.wolves_gain;
	const uint32_t sheep_thr = tr.sheep_thr, wolves_thr = tr.wolves_thr, R = tr.R;
	GT *s_g = reinterpret_cast<GT *>(s_grass);
	/* x and row of a cell index */
	auto cell_xr = [&](uint32_t c, uint32_t &x, uint32_t &r) {
		if (D2) {
			r = c >> tr.shift;
			x = c & (g.pitch - 1);
		} else {
			r = div_by(c, tr.gxm, tr.gxs);
			x = c - r * gx;
		}
	};
	uint32_t eaten = 0, ovf = 0;
	{
		const uint32_t nlist = s_nlist;
#pragma unroll 1
		for (uint32_t i = NT - 1 - tid; i < nlist; i += NT) {
			const uint32_t p = s_list[i], c = s_cell[p + 1];
			uint32_t kk = s_start[c + 1] - p, cl;
			if (D2) {
				uint32_t x, r;
				cell_xr(c, x, r);
				cl = (g.y0 + r) * gx + g.x0 + x;
			} else {
				cl = g.y0 * gx + c;
			}
			const bool alive = grass_alive_at<GT>(s_g[c], tick + 1, P.R);
			bool ate;
			if (kk <= 4)
				ate = tile_cell<4>(s_val, s_id, p, kk, alive, cl, step, key0, key1,
					sheep_gain, wolves_gain, sheep_thr, wolves_thr, &ovf);
			else if (kk <= 8)
				ate = tile_cell<8>(s_val, s_id, p, kk, alive, cl, step, key0, key1,
					sheep_gain, wolves_gain, sheep_thr, wolves_thr, &ovf);
			else
				ate = tile_cell_any(s_val, s_id, p, kk, alive, cl, step, key0, key1,
					sheep_gain, wolves_gain, sheep_thr, wolves_thr, &ovf);
			if (ate) {
				s_g[c] = (GT)(tick + 1 + R);
				eaten++;
			}
		}
	}
	/* (this loop and those below are not unrolled: a group runs through the
	 * code about once, and fetching instructions is then what takes the time) */
#pragma unroll 1
	for (uint32_t p = tid; p < L; p += NT) {
		const uint32_t c = s_cell[p + 1];
		if (s_cell[p] == c || s_cell[p + 2] == c) continue;
		eaten += 1u << 16;     /* high half: these cells */
		const uint32_t v = s_val[p];
		int32_t e = (int32_t)(v & V_ENERGY);
		uint32_t thr = wolves_thr;
		if (!(v & V_WOLF)) {
			thr = sheep_thr;
			if (grass_alive_at<GT>(s_g[c], tick + 1, P.R)) {
				e += (int32_t)sheep_gain;
				s_g[c] = (GT)(tick + 1 + R);
				eaten++;
			}
		}
		uint32_t nv = v & V_WOLF;
		if (e > (int32_t)thr && (v & V_REPRO)) {
			nv |= V_CHILD | ((e & 1) ? V_ODD : 0u);
			e -= e / 2;
		}
		if (e > (int32_t)V_ENERGY) ovf = 1;
		s_val[p] = nv | ((uint32_t)e & V_ENERGY);
	}
	if (ovf) s_ovf = 1;
	__syncthreads();

	/* 4. the outputs of each slot and their offsets: slot order is (j, wave,
	 * lane), so ballots give the place in the wave and one scan over the
	 * waves' counts the rest */
	uint32_t n_all = 0, n_wolves = 0, e_all = 0, e_wolves = 0, n_birth = 0;
	const uint32_t rounds = (L + NT - 1) / NT;
#pragma unroll 1
	for (uint32_t j = 0; j < rounds; j++) {
		const uint32_t p = j * NT + tid;
		const uint32_t v = p < L ? s_val[p] : V_KILLED;
		const bool surv = !(v & V_KILLED), child = (v & V_CHILD) != 0;
		const bool wolf = (v & V_WOLF) != 0;
		const uint64_t bs = __ballot(surv), bc = __ballot(child), bw = __ballot(wolf);
		const uint32_t nb = (uint32_t)__popcll(bc), n = nb + (uint32_t)__popcll(bs);
		if (lane == 0) s_wt[j * NW + w] = n;
		n_all += n;
		n_birth += nb;
		n_wolves += (uint32_t)(__popcll(bs & bw) + __popcll(bc & bw));
		const uint32_t e = v & V_ENERGY;
		const uint32_t en = (surv ? e : 0u) + (child ? e - ((v & V_ODD) ? 1u : 0u) : 0u);
		e_all += en;
		e_wolves += wolf ? en : 0u;
	}
	{
		const uint32_t ne = wave_sum32(eaten);
		unsigned long long ea, ew;
		/* (a lane's sums stay below 2^(24 + 5)) */
		if (__ballot((e_all >> 26) != 0) == 0) {
			ea = wave_sum32(e_all);
			ew = wave_sum32(e_wolves);
		} else {
			ea = wave_sum((unsigned long long)e_all);
			ew = wave_sum((unsigned long long)e_wolves);
		}
		if (lane == 0) {
			s_red[w][0] = n_all - n_wolves;
			s_red[w][1] = n_wolves;
			s_red[w][2] = ne & 0xFFFFu;
			s_red[w][3] = (ne >> 16) + (w == 0 ? s_nlist : 0u);
			s_red[w][4] = n_birth;
			s_red[w][5] = w == 0 ? L : 0u;
			s_red[w][6] = ea - ew;
			s_red[w][7] = ew;
		}
	}
	__syncthreads();
	const uint32_t wt = s_wt[NWT * lane], wt2 = NWT == 2 ? s_wt[2 * lane + 1] : 0u;
	const uint32_t wi = wave_incl_scan32(wt + wt2);
	const uint32_t nout = (uint32_t)__builtin_amdgcn_readlane((int)wi, WAVE - 1);
	uint32_t o_at = tile * A.slot, o_max = nout;
	if (nout > A.slot) {
		if (tid == 0) s_tmp[0] = atomicAdd(&A.spare[1 - A.par], nout);
		__syncthreads();
		const uint32_t q = s_tmp[0];
		/* (past the spare records only with more agents than the capacity:
		 * the batch then fails, and nothing is written) */
		if (q + nout > P.cap) o_max = 0;
		o_at = A.spare0 + (o_max ? q : 0u);
	}
	o_at = __builtin_amdgcn_readfirstlane(o_at);
	uint2 *o_rec = A.out + o_at;
	uint2 *o_edge = D2 ? A.eout + 2 * TILE_ECAP * tile : nullptr;
#pragma unroll 1
	for (uint32_t j = 0; j < rounds; j++) {
		const uint32_t p = j * NT + tid;
		const bool in = p < L;
		const uint32_t v = in ? s_val[p] : V_KILLED;
		const uint64_t bs = __ballot(!(v & V_KILLED)), bc = __ballot((v & V_CHILD) != 0);
		uint32_t o = __builtin_amdgcn_mbcnt_hi((uint32_t)(bs >> 32),
			__builtin_amdgcn_mbcnt_lo((uint32_t)bs,
			__builtin_amdgcn_mbcnt_hi((uint32_t)(bc >> 32),
			__builtin_amdgcn_mbcnt_lo((uint32_t)bc, 0u))));
		const uint32_t jw = j * NW + w;
		o += (uint32_t)__builtin_amdgcn_readlane((int)(wi - wt - wt2), (int)(jw / NWT));
		if (NWT == 2 && (jw & 1u))
			o += (uint32_t)__builtin_amdgcn_readlane((int)wt, (int)(jw / 2));
		if (!in) continue;
		s_id[p] = o;   /* (the ids are no longer needed) */
		uint32_t x, r;
		cell_xr(s_cell[p + 1], x, r);
		const uint32_t rx = x | (r << 16);
		const uint32_t y = v & (V_ENERGY | V_WOLF);
		auto put = [&](uint32_t y) {
			if (o < o_max) at32(o_rec, o) = make_uint2(rx, y);
			if (D2 && !wrapx) {
				/* edge lists of the neighbours left and right */
				const uint2 er = make_uint2(o | (r << 16), y);
				if (x == 0) {
					const uint32_t q = atomicAdd(&s_edge[0], 1u);
					if (q < TILE_ECAP) o_edge[q] = er;
				}
				if (x == g.w - 1) {
					const uint32_t q = atomicAdd(&s_edge[1], 1u);
					if (q < TILE_ECAP) o_edge[TILE_ECAP + q] = er;
				}
			}
			o++;
		};
		if (!(v & V_KILLED)) put(y);
		if (v & V_CHILD) put(y - ((v & V_ODD) ? 1u : 0u));
	}
	/* the grass back; alive cells are re-stamped now and then (see REFRESH),
	 * with this tick, so that they are alive in it also where it fails */
	const bool restamp = tick % TILE_RESTAMP == 0;
#pragma unroll 1
	for (uint32_t i = tid; i < CHUNKS; i += NT) {
		uint32_t cell, cells;
		if (!G.chunk(i, cell, cells)) continue;
		if (restamp) {
			GT *q = s_g + i * TG::VPC;
#pragma unroll 1
			for (uint32_t u = 0; u < TG::VPC; u++)
				if (grass_alive_at<GT>(q[u], tick + 1, P.R) && q[u] != (GT)(tick + 1))
					q[u] = (GT)tick;
		}
		if (cells >= TG::VPC) {
			const uint4 v = s_grass[i];
			*reinterpret_cast<Grass16 *>(grass + cell) = Grass16{{v.x, v.y, v.z, v.w}};
		} else {
			for (uint32_t u = 0; u < cells; u++) grass[cell + u] = s_g[i * TG::VPC + u];
		}
	}
	__syncthreads();
	/* first record of each row (the output offset of the row's first slot) */
	auto row_first = [&](uint32_t r) {
		const uint32_t q = s_row[D2 ? r : r == 1 && g.h > 2 ? 0u : 1u];
		return q < L ? s_id[q] : nout;
	};
	if (D2)
		for (uint32_t r = tid; r <= g.h; r += NT)
			A.rout[(size_t)tile * (A.rows + 1) + r] = r < g.h ? row_first(r) : nout;
	if (tid < 8) {
		unsigned long long v = 0;
#pragma unroll 4
		for (uint32_t i = 0; i < NW; i++) v += s_red[i][tid];
		A.sout[tile].v[tid] = v;
	}
	if (tid == 0) {
		const uint32_t nf = g.h > 1 ? row_first(1) : nout;
		const uint32_t nla = g.h > 1 ? nout - row_first(g.h - 1) : nout;
		const uint32_t el = D2 ? s_edge[0] : 0u, er = D2 ? s_edge[1] : 0u;
		A.hout[tile] = make_uint4(nout, nf | (nla << 16), min(el, TILE_ECAP) |
			(min(er, TILE_ECAP) << 16), o_at);
		if (nout > A.nmax || nf > A.hmax || nla > A.hmax || el > TILE_ECAP ||
			er > TILE_ECAP)
			ctl->stop = tick + 2;
		if (s_ovf) T.rctl[tr.slot].ovf = tick + 1;
		if (!SOLO)
			atomicAdd(&A.tot[(tick % 3) * PART_SLOTS + tile % PART_SLOTS],
				(unsigned long long)nout);
		if (D2)
			atomicAdd(&A.bsum[(1 - A.par) * A.nbands + tr.band0 + lt / tr.nbx], nout);
	}
}

/* After an iteration of tiles that cut grid rows (D2): one work-group per
 * band (row of tiles) turns the agents per tile row into ids: the bands
 * before it, then a scan over the band's rows, tile by tile; also the band's
 * statistics, and the replica's agents (last band). A chain of memory round
 * trips: what can be requested together is, and a thread takes four tile rows
 * in turn (12800 x 12800: 11.4 -> 9.6 us, 4001 x 2999 5.5 -> 5.0, with its
 * iteration 46.6 -> 45.3). again: for a state whose ids the scan after a
 * failed tick has replaced, its bands' sums by k_tile_bands. */
__global__ __launch_bounds__(WG) void k_tile_scan(TileArgs A, Ctl *ctl,
	Params P, uint32_t nrep, uint32_t again) {
	const bool SOLO = nrep == 1;
	constexpr uint32_t EPT = 4;
	__shared__ uint32_t s_tmp[NWAVE];
	__shared__ unsigned long long s_f[NWAVE][8];
	/* only after a tick that ran */
	if (!again && (ctl->error || ctl->halt || ctl->tt[1 - A.par] != ctl->tt[A.par] + 1))
		return;
	if (again && !ctl->records) return;
	const uint32_t band = blockIdx.x, tid = threadIdx.x;
	const uint32_t k = nrep == 1 ? 0u : A.bk[band];
	const TileRep tr = SOLO ? A.one : tile_rep(A.trep, k);
	const uint32_t ty = band - tr.band0;
	const uint32_t n = min(tr.by, tr.gy - ty * tr.by) * tr.nbx;
	const uint32_t *bs = A.bsum + (1 - A.par) * A.nbands + tr.band0;
	const uint32_t t0 = tr.tile0 + ty * tr.nbx;
	uint32_t base = 0, tot;
	for (uint32_t i = tid; i < ty; i += WG) base += bs[i];
	for (uint32_t e0 = 0; e0 < n; e0 += WG * EPT) {
		/* EPT rows of tiles a thread, one after another */
		uint32_t first[EPT], cnt[EPT], at[EPT], sum = 0;
#pragma unroll
		for (uint32_t i = 0; i < EPT; i++) {
			const uint32_t e = min(e0 + tid * EPT + i, n - 1), r = e / tr.nbx;
			const uint32_t t = t0 + (e - r * tr.nbx);
			const uint32_t *rs = A.rout + (size_t)t * (A.rows + 1) + r;
			at[i] = t * A.rows + r;
			first[i] = rs[0];
			cnt[i] = e0 + tid * EPT + i < n ? rs[1] - first[i] : 0u;
			sum += cnt[i];
		}
		if (e0 == 0) {
			/* (the bands' sums and the first rows are requested together) */
			(void)wg_excl_scan<WG>(base, s_tmp, tot);
			base = tot;
		}
		uint32_t x = base + wg_excl_scan<WG>(sum, s_tmp, tot);
#pragma unroll
		for (uint32_t i = 0; i < EPT; i++) {
			if (e0 + tid * EPT + i < n) A.idoff[at[i]] = x - first[i];
			x += cnt[i];
		}
		base += tot;
	}
	if (tid == 0) {
		if (ty + 1 == tr.nby) A.rtot[k] = base;
		A.bsum[A.par * A.nbands + band] = 0;
	}
	/* more agents than the capacity: no tick runs on them (see k_tile) */
	if (!SOLO && band == 0 && tid < WAVE) {
		const uint32_t t = ctl->tt[A.par] % 3;
		if (wave_sum32((uint32_t)A.tot[t * PART_SLOTS + tid]) > P.cap && tid == 0)
			ctl->halt = 1;
	}
	stat_sums<WG>(A.sout + t0, tr.nbx, s_f);
	if (tid < 8) {
		unsigned long long a = 0;
		for (int q = 0; q < NWAVE; q++) a += s_f[q][tid];
		A.bstat[band].v[tid] = a;
	}
}

/* The agents of each band, of the tiles in A.hout. */
__global__ __launch_bounds__(WG) void k_tile_bands(TileArgs A, const Ctl *ctl,
	uint32_t nrep) {
	__shared__ uint32_t s_tmp[NWAVE];
	if (!ctl->records) return;
	const uint32_t band = blockIdx.x, tid = threadIdx.x;
	const TileRep tr = nrep == 1 ? A.one : tile_rep(A.trep, A.bk[band]);
	const uint32_t t0 = tr.tile0 + (band - tr.band0) * tr.nbx;
	uint32_t sum = 0, tot;
	for (uint32_t i = tid; i < tr.nbx; i += WG) sum += A.hout[t0 + i].x;
	(void)wg_excl_scan<WG>(sum, s_tmp, tot);
	if (tid == 0) A.bsum[(1 - A.par) * A.nbands + band] = tot;
}

/* The end of the last tick run, one work-group per replica of the table. A
 * holds the buffers by parity: in/hin/sin parity 0, out/hout/sout parity 1. */
template <bool D2>
__global__ __launch_bounds__(WG) void k_tile_end(TileArgs A, Ctl *ctl, Tables T,
	Params P, uint32_t nrep) {
	const bool SOLO = nrep == 1;
	if (ctl->error) return;
	const uint32_t cur = tile_last(ctl), tick = ctl->tt[cur], k = blockIdx.x;
	const TileRep tr = SOLO ? A.one : tile_rep(A.trep, k);
	const TileStat *st = cur ? A.sout : A.sin;
	tile_finish<WG>(D2 ? A.bstat + tr.band0 : st + tr.tile0,
		D2 ? tr.nby : tr.ntiles, k, tick - 1, A.tot, ctl, T, P, nrep);
}

/* Batch positions of the replicas' agents, in table order (the SoA state),
 * and their number. One wave. */
__global__ __launch_bounds__(WAVE) void k_tile_base(Ctl *ctl, Tables T,
	uint32_t nrep) {
	const uint32_t lane = threadIdx.x;
	uint32_t carry = 0;
	if (!ctl->records) return;
	for (uint32_t k0 = 0; k0 < nrep; k0 += WAVE) {
		const uint32_t k = k0 + lane;
		uint32_t n = 0, slot = 0;
		if (k < nrep) {
			slot = T.order[k];
			n = T.rctl[slot].status == RS_ACTIVE ? T.rctl[slot].n : 0u;
		}
		const uint32_t x = wave_incl_scan32(n);
		if (k < nrep) T.rctl[slot].base = carry + x - n;
		carry += (uint32_t)__builtin_amdgcn_readlane((int)x, WAVE - 1);
	}
	if (lane == 0) ctl->n = carry;
}

/* Before k_tiles_in: no records, no stop, and the bands' sums (both parities)
 * at zero. */
__global__ __launch_bounds__(WG) void k_tile_clear(TileArgs A, Ctl *ctl) {
	const uint32_t i = blockIdx.x * WG + threadIdx.x;
	if (i == 0) ctl->stop = ctl->halt = ctl->records = 0;
	if (i < 2) A.spare[i] = 0;
	if (i < 2 * A.nbands) A.bsum[i] = 0;
}

/* Re-stamps a tile's alive cells with the tick (see REFRESH), by chunks. */
template <typename GT, bool D2>
__device__ __forceinline__ void tile_restamp(const TileGrass<GT, D2> &G, GT *grass,
	uint32_t tick, uint32_t R) {
	using TG = TileGrass<GT, D2>;
	const uint32_t chunks = D2 ? G.rows << G.csh : (G.n + TG::VPC - 1) / TG::VPC;
	for (uint32_t i = threadIdx.x; i < chunks; i += WG) {
		uint32_t cell, cells;
		if (!G.chunk(i, cell, cells)) continue;
		GT v[TG::VPC];
		if (cells >= TG::VPC) {
			__builtin_memcpy(v, grass + cell, 16);
#pragma unroll
			for (uint32_t u = 0; u < TG::VPC; u++)
				if (grass_alive_at<GT>(v[u], tick, R)) v[u] = (GT)tick;
			__builtin_memcpy(grass + cell, v, 16);
		} else {
			for (uint32_t u = 0; u < cells; u++)
				if (grass_alive_at<GT>(grass[cell + u], tick, R))
					grass[cell + u] = (GT)tick;
		}
	}
}

/* The first of n ascending values that is not below c, by LANES lanes that
 * hold the same arguments (a whole aligned group of a wave): each trip to
 * memory leaves one of LANES + 1 parts. (One lane's binary search of 42 M
 * agents took 26 trips, two of them in turn for each row of a tile: 0.9 ms of
 * k_tiles_in's 1.0 at 12800 x 12800.) */
template <uint32_t LANES>
__device__ __forceinline__ uint32_t lower_by(const uint32_t *a, uint32_t n, uint32_t c) {
	const uint32_t lane = threadIdx.x & (WAVE - 1), j = lane % LANES;
	uint32_t lo = 0, hi = n;
	while (lo < hi) {
		const uint64_t len = hi - lo;
		const uint32_t mid = lo + (uint32_t)(len * (j + 1) / (LANES + 1));
		uint64_t below = __ballot(a[mid] < c) >> (lane - j);
		if (LANES < WAVE) below &= (1ull << (LANES % WAVE)) - 1;
		const uint32_t q = (uint32_t)__popcll(below);
		hi = q < LANES ? lo + (uint32_t)(len * (q + 1) / (LANES + 1)) : hi;
		lo = q ? lo + (uint32_t)(len * q / (LANES + 1)) + 1 : lo;
	}
	return lo;
}

/* The SoA state (sorted by cell within each replica) into the tiles' slots
 * (parity 0). */
template <typename GT, bool D2>
__global__ __launch_bounds__(WG) void k_tiles_in(TileArgs A, Ctl *ctl, Tables T,
	Params P, uint32_t nrep, GT *grass, const uint32_t *cell,
	const int32_t *energy, const uint8_t *type) {
	const bool SOLO = nrep == 1;
	__shared__ uint32_t s_lo[D2 ? TILE_ROWS : 1], s_n[D2 ? TILE_ROWS + 1 : 1];
	__shared__ uint32_t s_b[4], s_edge[2];
	if (ctl->error) return;
	const uint32_t tid = threadIdx.x, tile = blockIdx.x, tick = ctl->tick;
	if (tile == 0) {
		if (tid == 0) {
			ctl->tt[0] = tick;
			ctl->tt[1] = tick - 1;
			ctl->in_tick = tick;
			ctl->records = 1;
		}
		if (tid < PART_SLOTS)
			for (uint32_t i = 0; i < 3; i++) A.tot[i * PART_SLOTS + tid] = 0;
	}
	const uint32_t k = nrep == 1 ? 0u : A.tk[tile];
	const uint32_t slot = T.order[k];
	const Rep &rp = T.rep[slot];
	const RepCtl &rc = T.rctl[slot];
	const TileRep tr = SOLO ? A.one : tile_rep(A.trep, k);
	const TileGeo g = tile_geo<D2>(tr, tile - tr.tile0, rp.gx, rp.gy);
	const uint32_t base = rc.base, n = rc.status == RS_ACTIVE ? rc.n : 0u;
	const TileGrass<GT, D2> G(rp.cb + g.y0 * rp.gx + g.x0, rp.gx, g.w, g.h, tr.shift);
	uint2 *o_edge = D2 ? const_cast<uint2 *>(A.ein) + 2 * TILE_ECAP * tile : nullptr;
	if (tid < 2) s_edge[tid] = 0;
	uint32_t nout, nf, nl;
	/* the slot, or spare records, for nout agents (a tile above the limits
	 * keeps none of them: the SoA state stays the valid one) */
	auto place = [&](uint32_t n_) {
		if (tid == 0) {
			uint32_t q = tile * A.slot;
			if (n_ > A.slot && n_ <= A.nmax) q = A.spare0 + atomicAdd(&A.spare[0], n_);
			s_b[0] = q;
		}
		__syncthreads();
		return s_b[0];
	};
	uint32_t o_at;
	if (!D2) {
		/* row bounds of the tile, its second and its last row */
		static_assert(WG / WAVE == 4, "a wave for each bound");
		const uint32_t q = tid / WAVE;
		const uint32_t r = q == 0 ? 0u : q == 1 ? 1u : q == 2 ? g.h - 1 : g.h;
		const uint32_t at = lower_by<WAVE>(cell + base, n, rp.cb + (g.y0 + r) * rp.gx);
		if (tid % WAVE == 0) s_b[q] = at;
		__syncthreads();
		nout = s_b[3] - s_b[0];
		nf = s_b[1] - s_b[0];
		nl = s_b[3] - s_b[2];
		const uint32_t lo = s_b[0], take = nout > A.nmax ? 0u : nout;
		__syncthreads();
		o_at = place(nout);
		uint2 *o_rec = const_cast<uint2 *>(A.in) + o_at;
		const uint32_t c0 = rp.cb + g.y0 * rp.gx;
		for (uint32_t i = tid; i < take; i += WG) {
			const uint32_t p = base + lo + i, c = cell[p] - c0;
			const uint32_t r = c / rp.gx, x = c - r * rp.gx;
			o_rec[i] = make_uint2(x | (r << 16),
				(uint32_t)energy[p] | (type[p] ? V_WOLF : 0u));
		}
		tile_restamp(G, grass, tick, P.R);
	} else {
		/* first agents of the rows (even q) and of what follows them */
		for (uint32_t q0 = 0; q0 < 2 * g.h; q0 += WG / 8) {
			const uint32_t q = q0 + tid / 8, r = q / 2;
			if (r >= g.h) break;
			const uint32_t c = rp.cb + (g.y0 + r) * rp.gx + g.x0 + (q & 1u ? g.w : 0u);
			const uint32_t at = lower_by<8>(cell + base, n, c);
			if (tid % 8 == 0) (q & 1u ? s_n[r + 1] : s_lo[r]) = at;
		}
		__syncthreads();
		if (tid == 0) {
			s_n[0] = 0;
			for (uint32_t r = 0; r < g.h; r++) s_n[r + 1] = s_n[r] + s_n[r + 1] - s_lo[r];
		}
		__syncthreads();
		nout = s_n[g.h];
		nf = s_n[1];
		nl = nout - s_n[g.h - 1];
		o_at = place(nout);
		uint2 *o_rec = const_cast<uint2 *>(A.in) + o_at;
		for (uint32_t r = tid; r <= g.h; r += WG)
			const_cast<uint32_t *>(A.rin)[(size_t)tile * (A.rows + 1) + r] = s_n[r];
		/* a wave to a row, whose agents are about as many as its lanes */
		for (uint32_t r = tid / WAVE; r < g.h; r += WG / WAVE) {
			const uint32_t c0 = rp.cb + (g.y0 + r) * rp.gx + g.x0;
			for (uint32_t i = tid % WAVE; i < s_n[r + 1] - s_n[r]; i += WAVE) {
				const uint32_t o = s_n[r] + i;
				if (nout > A.nmax) break;
				const uint32_t p = base + s_lo[r] + i, x = cell[p] - c0;
				const uint32_t y = (uint32_t)energy[p] | (type[p] ? V_WOLF : 0u);
				o_rec[o] = make_uint2(x | (r << 16), y);
				if (tr.nbx > 1) {
					const uint2 er = make_uint2(o | (r << 16), y);
					if (x == 0) {
						const uint32_t q = atomicAdd(&s_edge[0], 1u);
						if (q < TILE_ECAP) o_edge[q] = er;
					}
					if (x == g.w - 1) {
						const uint32_t q = atomicAdd(&s_edge[1], 1u);
						if (q < TILE_ECAP) o_edge[TILE_ECAP + q] = er;
					}
				}
			}
		}
		tile_restamp(G, grass, tick, P.R);
		__syncthreads();
		if (tid == 0)
			atomicAdd(&A.bsum[tr.band0 + (tile - tr.tile0) / tr.nbx], nout);
	}
	if (tid == 0) {
		const uint32_t el = D2 ? s_edge[0] : 0u, er = D2 ? s_edge[1] : 0u;
		const_cast<uint4 *>(A.hin)[tile] = make_uint4(nout, nf | (nl << 16),
			min(el, TILE_ECAP) | (min(er, TILE_ECAP) << 16), o_at);
		if (nout > A.nmax || nf > A.hmax || nl > A.hmax || el > TILE_ECAP ||
			er > TILE_ECAP)
			ctl->stop = tick + 1;
	}
}

/* The tiles' records (of Ctl::tick, also after an iteration that failed the
 * batch) to the SoA state, at the replicas' batch positions (k_tile_base), and
 * their grass re-stamped. A holds the buffers by parity, as for k_tile_end. */
template <typename GT, bool D2>
__global__ __launch_bounds__(WG) void k_tiles_out(TileArgs A, Ctl *ctl, Tables T,
	Params P, uint32_t nrep, GT *grass, uint32_t *cell, int32_t *energy,
	uint8_t *type) {
	const bool SOLO = nrep == 1;
	__shared__ uint32_t s_tmp[NWAVE];
	const uint32_t tid = threadIdx.x, tile = blockIdx.x;
	if (!ctl->records) return;
	const uint32_t cur = tile_cur(ctl), tick = ctl->tick;
	const uint32_t k = nrep == 1 ? 0u : A.tk[tile];
	const uint32_t slot = T.order[k];
	const Rep &rp = T.rep[slot];
	const RepCtl &rc = T.rctl[slot];
	if (rc.status != RS_ACTIVE) return;
	const TileRep tr = SOLO ? A.one : tile_rep(A.trep, k);
	const uint32_t lt = tile - tr.tile0;
	const TileGeo g = tile_geo<D2>(tr, lt, rp.gx, rp.gy);
	const uint4 *hdr = cur ? A.hout : A.hin;
	uint32_t idb = 0;
	if (!D2) {
		uint32_t sum = 0;
		for (uint32_t i = tid; i < lt; i += WG) sum += hdr[tr.tile0 + i].x;
		(void)wg_excl_scan<WG>(sum, s_tmp, idb);
	}
	const uint2 *recs = (cur ? A.out : A.in) + hdr[tile].w;
	const uint32_t n = hdr[tile].x;
	for (uint32_t i = tid; i < n; i += WG) {
		const uint2 q = recs[i];
		const uint32_t x = q.x & 0xFFFFu, r = q.x >> 16;
		const uint32_t id = rc.base + i + (D2 ? A.idoff[tile * A.rows + r] : idb);
		if (id >= P.cap) continue;
		cell[id] = rp.cb + (g.y0 + r) * rp.gx + g.x0 + x;
		energy[id] = (int32_t)(q.y & V_ENERGY);
		type[id] = (q.y & V_WOLF) ? PP_WOLF : PP_SHEEP;
	}
	const TileGrass<GT, D2> G(rp.cb + g.y0 * rp.gx + g.x0, rp.gx, g.w, g.h, tr.shift);
	tile_restamp(G, grass, tick, P.R);
}
