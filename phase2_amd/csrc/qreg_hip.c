/*
 * BACKEND=hip register (replaces phase2/qreg.c, phase2/qreg_qreg.c and
 * phase2/qreg_cuda.c of the reference on one GPU).
 *
 * One hipMalloc buffer holds the whole register; with one process there is
 * no hi/lo split (qb_hi = 0), no partner exchange and no mix/add passes:
 * the reference's single-rank flush (self-exchange, mix with bm = 1, rotate,
 * add 0) reduces exactly to in-order rotations, which is what
 * qreg_paulirot applies here.  cos/sin come from the host libm per term as
 * in phase2/qreg_qreg.c:189, through sincos(): gcc folds the reference's
 * adjacent cos() and sin() of one angle into a single glibc sincos() call,
 * whose results differ from separate cos()/sin() calls by one ulp for some
 * angles, so calling sincos() explicitly is what reproduces the reference.
 *
 * The void entry points cannot return errors; a failed device call logs
 * and sets a sticky flag read by qreg_error().
 */
#define _GNU_SOURCE /* sincos */
#define LOG_SUBSYS "qreg"

#include <complex.h>
#include <math.h>
#include <stdlib.h>
#include <string.h>

#include "log.h"
#include "phase2/qreg.h"
#include "phase2/qreg_hip.h"
#include "phase2/world.h"
#include "phase2_hip.h"

/* A block of rotations as the register last saw it: its codes and angles,
 * and from them the rotations with their sines and cosines and the greedy
 * schedule.  A Trotter step applies the same blocks every step; for 1024
 * terms the sines take 15 us and the schedule 10, and the device of a
 * narrow register waits for them. */
#define BLOCKS 8
#define BLOCK_MAX 4096	/* larger ones share the first slot */
struct block {
	size_t n, cap;
	struct paulis *codes;
	double *phis;
	struct ph2hip_rot *rot;
	struct ph2_sched sched;
	int scheduled;	/* sched is the greedy one of the settings below */
	int chosen;	/* the tile and low bits are automatic */
	uint32_t tile, low, half;	/* low as asked for */
	uint64_t used;
};

struct qreg_hip {
	void *damp;
	int err;
	int mode;
	uint32_t tile_bits, low_bits;
	struct block blocks[BLOCKS];	/* least recently used out */
	uint64_t clock;
	struct ph2_sched sched;		/* of a schedule function */
	/* state a caller above the register keeps with it (the multidet
	 * overlap plan of circ.c), released by qreg_free */
	void *aux;
	void (*aux_free)(void *);
	/* qreg_setamp writes not yet on the device, in call order */
	uint64_t *qidx;
	double *qval;
	size_t nq, qcap;
	int pending;	/* work on the buffer sent to the stream and not waited
			 * for since: SENT_WRITES, SENT_WORK */
	/* host copy of amplitudes [win_lo, win_lo + win_n) as the device
	 * holds them with the queued writes applied; win_n = 0: none */
	double *win;
	uint64_t win_lo, win_n;
	/* reads since the buffer last changed: the first one's window, whether
	 * others left it; and whether they did between the two changes before */
	uint64_t first_lo;
	int reads, spread, wide;
};

/* One amplitude moved by itself costs a synchronous device copy (about
 * 10 µs), so a loop over a register's amplitudes through qreg_setamp /
 * qreg_getamp, as the reference's callers and tests write, would run at
 * 10^5 amplitudes per second.  Writes are queued on the host and land in
 * one scatter (later writes to an index win) before anything else touches
 * the device buffer; reads are served from a host copy of an aligned
 * window, taken after the queue has landed, kept current by later
 * qreg_setamp calls and dropped by every operation that may change the
 * buffer.  AMP_WIN amplitudes cost 30 us to fetch, AMP_FIRST through pinned
 * memory little more than one alone (11 us), and often one is all that is
 * read between two changes: the first read after a change takes AMP_FIRST,
 * one outside them AMP_WIN, and where reads spread like that the next change
 * is followed by AMP_WIN at once. */
#define AMP_WIN (UINT64_C(1) << 14)  /* 256 KiB */
#define AMP_FIRST (UINT64_C(1) << 10)
#define AMP_QMAX ((size_t)1 << 20)   /* 24 MiB of queued writes */

#define SENT_WRITES 1
#define SENT_WORK 2

static int g_mode = -1;
/* tile 0: auto_tile(), with low 3 auto_low() */
static uint32_t g_tile = 0, g_low = 3;
static ph2_sched_fn g_sched_fn;
static void *g_sched_ctx;

/* Tile width when none is set, from 1024-term blocks timed at every tile
 * width, lex-ordered sweeps and random draws at low bits 2 (us per block,
 * sweep / draw; settings in turn, median of seven):
 *   to 18 qubits, tile 10: 351 / 373 at 16 qubits and 411 / 458 at 18
 *     against 384 / 416 and 432 / 486 at tile 11, 119 / 198 against 155 /
 *     245 at tile 9 at 10 qubits.  A few dozen workgroups, bound by each
 *     pass's chain of terms and exchanges;
 *   19 to 21, tile 11: 680 / 862 at 20 and 998 / 945 at 21 against
 *     774 / 909 and 1221 / 1036 at tile 10, 751 / 907 and 1045 / 1002 at 12;
 *   from 22, tile 13: 1768 / 1497 at 22, 6664 / 4919 at 24, 14922 / 9928 at
 *     25, 125907 / 76237 at 28 against 1757 / 1529, 6973 / 4928, 16880 /
 *     10136 and 141426 / 78530 at tile 12.  Traffic per pass weighs most and
 *     wider tiles need fewer passes; at 22 the two are even.
 * Without replay of captured sweeps (ph2hip_replay_max_qb, 20 qubits by
 * default): 12 from 17 qubits, nqb - 5 under that, as fitted when a launch
 * cost more than a pass of the kernels.  It no longer does: the widths above
 * are the faster ones there too (394 us at tile 10 against 411 at 11 for a
 * sweep at 16 qubits, 447 against 613 at 12 at 18, 701 at 11 against 766 at
 * 12 at 20). */
static uint32_t auto_tile(uint32_t nqb)
{
	uint32_t t;
	if (nqb <= ph2hip_replay_max_qb()) {
		t = nqb >= 22 ? 13 : nqb >= 19 ? 11 : 10;
		if (t > nqb)
			t = nqb;
	} else {
		t = nqb >= 22 ? 13 : nqb == 21 ? 11 : nqb > 16 ? 12 :
			(nqb > 5 ? nqb - 5 : 0);
	}
	return t < PH2HIP_TILE_MIN ? PH2HIP_TILE_MIN : t;
}

/* Contiguous low bits the cut asks for under the automatic tile width: those
 * the caller set, but for the default (LOW_AUTO) 2, where rows of 64 bytes
 * leave one more dimension to gather than rows of 128.  Low 2 against 3:
 * random draws 373 and 401 us at 16 qubits, 458 and 502 at 18, 862 and 930
 * at 20; sweeps 351 and 353, 411 and 420, 680 and 680; 6664 and 6745 at 24,
 * 125907 and 130379 at 28.  Low 1 is slower from 30. */
#define LOW_AUTO 3
static uint32_t auto_low(uint32_t low)
{
	return low == LOW_AUTO ? 2 : low;
}

/* Under the automatic setting a block of a register of up to 18 or of 22 to 27
 * qubits is cut twice, and the number of passes says which cut it takes.
 *
 * To 18 qubits the state lies in the L2s, where short rows cost less than
 * passes: with no low bits asked for, sweeps (whose masks have an even
 * number of flips, so that single low bits are dimensions none of them
 * needs) take a third fewer passes and 328 us instead of 351 at 16 qubits,
 * 295 / 316 at 14, 394 / 411 at 18, but random draws a fifth fewer and 384
 * instead of 373, 401 / 378 and 479 / 458.  The second cut, without low
 * bits, is taken if it saves a quarter of the passes; to 12 qubits always
 * (276 / 286 and 218 / 225).  Low bits that the caller set stay.
 *
 * From 22 to 27 qubits a tile-12 pass is the shorter one: blocks of 1 to 40
 * terms that need as many passes at either width took 1.075, 1.078, 1.077,
 * 1.039, 1.018 and 1.030 times as long at tile 13 (22 to 27 qubits,
 * geometric mean of 17 to 23 blocks each, 0.99 at 28 and 1.01 at 29; a
 * setting timed twice, all in turn, differed by 0.1 to 0.6% in the mean).
 * Single blocks range from 0.87 to 1.32, and one of nine terms at 27 qubits
 * took 1331 us against 815.  The second cut, at tile 12, is taken unless
 * tile 13 saves a twentieth of its passes; blocks of 1024 terms save a
 * twelfth or more (at 22 qubits 41 passes instead of 45, 1497 us instead of
 * 1529). */
static int second_cut(uint32_t nqb, uint32_t asked, uint32_t *tile,
	uint32_t *low)
{
	if (nqb <= 18 && asked == LOW_AUTO)
		*low = 0;
	else if (nqb >= 22 && nqb <= 27 && *tile == 13)
		*tile = 12;
	else
		return 0;
	return 1;
}

static int take_second(uint32_t nqb, size_t first, size_t second)
{
	if (nqb <= 18)
		return nqb <= 12 || 4 * second <= 3 * first;
	return 20 * first > 19 * second;
}

static void load_defaults(void)
{
	if (g_mode >= 0)
		return;
	g_mode = QREG_HIP_FUSED;
	const char *m = getenv("PHASE2_HIP_MODE");
	if (m && strcmp(m, "plain") == 0)
		g_mode = QREG_HIP_PLAIN;
	const char *t = getenv("PHASE2_HIP_TILE");
	if (t) {
		const long v = strtol(t, NULL, 10);
		if (v >= PH2HIP_TILE_MIN && v <= PH2HIP_TILE_MAX)
			g_tile = (uint32_t)v;
	}
	const char *l = getenv("PHASE2_HIP_LOW");
	if (l) {
		const long v = strtol(l, NULL, 10);
		if (v >= 0 && v <= PH2HIP_TILE_MAX)
			g_low = (uint32_t)v;
	}
}

void qreg_hip_set_default(int mode, uint32_t tile_bits, uint32_t low_bits)
{
	load_defaults();
	g_mode = mode;
	g_tile = tile_bits;
	g_low = low_bits;
}

void qreg_hip_configure(struct qreg *reg, int mode, uint32_t tile_bits,
	uint32_t low_bits)
{
	struct qreg_hip *h = reg->backend;
	if (!h)
		return;
	h->mode = mode;
	h->tile_bits = tile_bits;
	h->low_bits = low_bits;
}

void ph2_sched_install(ph2_sched_fn fn, void *ctx)
{
	g_sched_fn = fn;
	g_sched_ctx = ctx;
}

/* Put the queued writes on the device: called before anything else reads or
 * changes the device buffer.  The read window holds them already. */
static int land(struct qreg_hip *h, uint64_t namp)
{
	if (h->nq == 0)
		return 0;
	const int rc = ph2hip_scatter_queue(h->damp, namp, h->qidx, h->qval,
		h->nq);
	h->nq = 0;
	h->pending |= SENT_WRITES;
	if (rc < 0) {
		h->err = -1;
		h->win_n = 0;
		log_error("qreg_setamp: %s", ph2hip_strerror());
	}
	return rc;
}

/* The buffer is about to change: the read window goes. */
static void forget(struct qreg_hip *h)
{
	h->win_n = 0;
	if (h->reads)
		h->wide = h->spread;
	h->reads = 0;
	h->spread = 0;
}

static int settle(struct qreg_hip *h, uint64_t namp)
{
	forget(h);
	return land(h, namp);
}

static void wait_pending(struct qreg_hip *h, const char *what)
{
	if (!h->pending)
		return;
	h->pending = 0;
	if (ph2hip_synchronize() < 0) {
		h->err = -1;
		log_error("%s: %s", what, ph2hip_strerror());
	}
}

/* For calls of this library, which queue their work behind the register's on
 * the same stream: the read window goes, and amplitude writes are waited for
 * once, so that their failure is known before a result is built on them.
 * The first overlap of a run therefore waits twice: 212 and 222 us for a
 * short call at 16 qubits without and with it, 2300 and 2287 at 24, where
 * hipFree of the register then takes 17 us instead of 330. */
void *qreg_hip_buffer(struct qreg *reg)
{
	struct qreg_hip *h = reg->backend;
	if (!h)
		return NULL;
	settle(h, reg->namp);
	if (h->pending & SENT_WRITES)
		wait_pending(h, "qreg_setamp");
	h->pending |= SENT_WORK;
	return h->damp;
}

/* The caller may read or change the buffer through the pointer on any
 * stream, so everything queued on it is done first: amplitude writes,
 * zeroing, rotations and the work of other calls of this library. */
void *qreg_hip_device_ptr(struct qreg *reg)
{
	struct qreg_hip *h = reg->backend;
	if (!h)
		return NULL;
	settle(h, reg->namp);
	wait_pending(h, "qreg_hip_device_ptr");
	return h->damp;
}

static void set_err(struct qreg *reg, const char *what)
{
	struct qreg_hip *h = reg->backend;
	if (h)
		h->err = -1;
	log_error("%s: %s", what, ph2hip_strerror());
}

int qreg_hip_send(struct qreg *reg)
{
	struct qreg_hip *h = reg->backend;
	if (!h)
		return -1;
	land(h, reg->namp);
	return h->err;
}

int qreg_error(const struct qreg *reg)
{
	struct qreg_hip *h = reg->backend;
	if (!h)
		return -1;
	/* a queued write fails, if at all, when it lands: land it now, and
	 * wait for it (short ones are only sent to the stream) */
	if (h->nq) {
		land(h, reg->namp);
		wait_pending(h, "qreg_error");
	}
	return h->err;
}

void qreg_clear_error(struct qreg *reg)
{
	struct qreg_hip *h = reg->backend;
	if (h)
		h->err = 0;
}

int qreg_init(struct qreg *reg, uint32_t qb)
{
	memset(reg, 0, sizeof *reg);
	if (world_info(&reg->wd) != WORLD_READY) {
		log_error("qreg_init: world not ready");
		return -1;
	}
	if (qb == 0 || qb > 40) {
		log_error("qreg_init: nqb=%u outside 1..40", qb);
		return -1;
	}
	load_defaults();
	struct qreg_hip *h = calloc(1, sizeof *h);
	if (!h) {
		log_error("qreg_init: alloc backend");
		return -1;
	}
	const uint64_t namp = UINT64_C(1) << qb;
	if (ph2hip_malloc(&h->damp, namp * 16) < 0) {
		log_error("qreg_init: device alloc of %llu bytes: %s",
			(unsigned long long)(namp * 16), ph2hip_strerror());
		free(h);
		return -1;
	}
	if (qb <= QREG_SHADOW_MAX_QB) {
		reg->amp = malloc(sizeof(_Complex double) * namp);
		if (!reg->amp) {
			log_error("qreg_init: host shadow alloc");
			ph2hip_free(h->damp);
			free(h);
			return -1;
		}
	}
	h->mode = g_mode;
	h->tile_bits = g_tile;
	h->low_bits = g_low;
	reg->qb_lo = qb;
	reg->qb_hi = 0;
	reg->buf = NULL;
	reg->namp = namp;
	reg->backend = h;
	return 0;
}

void *qreg_hip_aux(struct qreg *reg)
{
	const struct qreg_hip *h = reg->backend;
	return h ? h->aux : NULL;
}

int qreg_hip_set_aux(struct qreg *reg, void *aux, void (*aux_free)(void *))
{
	struct qreg_hip *h = reg->backend;
	if (!h)
		return -1;
	if (h->aux && h->aux_free)
		h->aux_free(h->aux);
	h->aux = aux;
	h->aux_free = aux_free;
	return 0;
}

void qreg_free(struct qreg *reg)
{
	struct qreg_hip *h = reg->backend;
	if (h) {
		if (h->aux && h->aux_free)
			h->aux_free(h->aux);
		ph2hip_free(h->damp);
		for (int i = 0; i < BLOCKS; i++) {
			free(h->blocks[i].codes);
			free(h->blocks[i].phis);
			free(h->blocks[i].rot);
			ph2_sched_free(&h->blocks[i].sched);
		}
		ph2_sched_free(&h->sched);
		free(h->qidx);
		free(h->qval);
		free(h->win);
		free(h);
	}
	free(reg->amp);
	reg->amp = NULL;
	reg->backend = NULL;
}

/* The reference masks an index to the register (phase2/qreg.c:35-47), so
 * on one rank an index beyond 2^qb silently aliases a lower one; here it is
 * an error (sticky flag, nothing read or written). */
static int in_range(struct qreg *reg, uint64_t i, const char *what)
{
	if (i < reg->namp)
		return 1;
	struct qreg_hip *h = reg->backend;
	h->err = -1;
	log_error("%s: index %llu beyond %u qubits", what,
		(unsigned long long)i, reg->qb_lo);
	return 0;
}

void qreg_getamp(struct qreg *reg, uint64_t i, _Complex double *z)
{
	struct qreg_hip *h = reg->backend;
	*z = 0.0;
	if (!in_range(reg, i, "qreg_getamp"))
		return;
	if (!h->win_n || i - h->win_lo >= h->win_n) {
		h->win_n = 0;
		if (land(h, reg->namp) < 0)
			return;
		if (!h->win && !(h->win = malloc((reg->namp < AMP_WIN ?
					reg->namp : AMP_WIN) * 16))) {
			log_error("qreg_getamp: alloc");
			h->err = -1;
			return;
		}
		const uint64_t size = h->reads || h->wide ? AMP_WIN : AMP_FIRST;
		const uint64_t lo = i & ~(size - 1);
		const uint64_t n = reg->namp - lo < size ? reg->namp - lo : size;
		if (ph2hip_read(h->damp, lo, n, h->win) < 0) {
			set_err(reg, "qreg_getamp");
			return;
		}
		h->win_lo = lo;
		h->win_n = n;
		if (!h->reads)
			h->first_lo = i & ~(AMP_FIRST - 1);
		h->reads = 1;
	}
	h->spread |= i - h->first_lo >= AMP_FIRST;
	const double *v = h->win + 2 * (i - h->win_lo);
	*z = CMPLX(v[0], v[1]);
}

void qreg_setamp(struct qreg *reg, uint64_t i, _Complex double z)
{
	struct qreg_hip *h = reg->backend;
	if (!in_range(reg, i, "qreg_setamp"))
		return;
	if (h->nq == h->qcap) {
		if (h->qcap >= AMP_QMAX) {
			if (land(h, reg->namp) < 0)
				return;
		} else {
			const size_t cap = h->qcap ? 2 * h->qcap : 1024;
			uint64_t *qi = realloc(h->qidx, sizeof *qi * cap);
			if (qi)
				h->qidx = qi;
			double *qv = realloc(h->qval, 2 * sizeof *qv * cap);
			if (qv)
				h->qval = qv;
			if (!qi || !qv) {
				log_error("qreg_setamp: alloc");
				h->err = -1;
				return;
			}
			h->qcap = cap;
		}
	}
	h->qidx[h->nq] = i;
	h->qval[2 * h->nq] = creal(z);
	h->qval[2 * h->nq + 1] = cimag(z);
	h->nq++;
	if (h->win_n && i - h->win_lo < h->win_n) {
		h->win[2 * (i - h->win_lo)] = creal(z);
		h->win[2 * (i - h->win_lo) + 1] = cimag(z);
	}
}

void qreg_zero(struct qreg *reg)
{
	struct qreg_hip *h = reg->backend;
	h->nq = 0; /* every queued write would be overwritten */
	forget(h);
	h->pending |= SENT_WORK;
	if (ph2hip_zero(h->damp, reg->namp) < 0)
		set_err(reg, "qreg_zero");
}

void qreg_sync_host_to_device(struct qreg *reg)
{
	struct qreg_hip *h = reg->backend;
	if (!reg->amp) {
		log_error("qreg_sync_host_to_device: no host shadow above %d "
			  "qubits", QREG_SHADOW_MAX_QB);
		h->err = -1;
		return;
	}
	h->nq = 0; /* every queued write would be overwritten */
	forget(h);
	if (ph2hip_h2d(h->damp, reg->amp, reg->namp * 16) < 0)
		set_err(reg, "qreg_sync_host_to_device");
}

void qreg_sync_device_to_host(struct qreg *reg)
{
	struct qreg_hip *h = reg->backend;
	if (!reg->amp) {
		log_error("qreg_sync_device_to_host: no host shadow above %d "
			  "qubits", QREG_SHADOW_MAX_QB);
		h->err = -1;
		return;
	}
	if (settle(h, reg->namp) < 0)
		return;
	if (ph2hip_d2h(reg->amp, h->damp, reg->namp * 16) < 0)
		set_err(reg, "qreg_sync_device_to_host");
}

/* The block of these codes and angles: an earlier one, compared in full, or
 * the least recently used one made theirs.  NULL: out of memory. */
static struct block *block_of(struct qreg_hip *h, const struct paulis *codes,
	const double *phis, size_t n)
{
	struct block *old = &h->blocks[0];
	for (int i = 0; i < BLOCKS; i++) {
		struct block *b = &h->blocks[i];
		if (b->used && b->n == n &&
		    memcmp(b->phis, phis, sizeof *phis * n) == 0 &&
		    memcmp(b->codes, codes, sizeof *codes * n) == 0) {
			b->used = ++h->clock;
			return b;
		}
		if (b->used < old->used)
			old = b;
	}
	if (n > BLOCK_MAX)
		old = &h->blocks[0];
	old->used = 0;
	old->scheduled = 0;
	if (n > old->cap) {
		free(old->codes);
		free(old->phis);
		free(old->rot);
		old->codes = malloc(sizeof *old->codes * n);
		old->phis = malloc(sizeof *old->phis * n);
		old->rot = malloc(sizeof *old->rot * n);
		old->cap = old->codes && old->phis && old->rot ? n : 0;
		if (!old->cap)
			return NULL;
	}
	memcpy(old->codes, codes, sizeof *codes * n);
	memcpy(old->phis, phis, sizeof *phis * n);
	for (size_t k = 0; k < n; k++) {
		old->rot[k].x = codes[k].pak[0];
		old->rot[k].z = codes[k].pak[1];
		sincos(phis[k], &old->rot[k].s, &old->rot[k].c);
	}
	old->n = n;
	old->used = ++h->clock;
	return old;
}

/* The fused sweep of a block: the schedule function's cut, else greedy. */
static int rotate_block(struct qreg_hip *h, uint32_t nqb, struct block *b)
{
	const struct ph2_sched *s = &h->sched;
	int rc = -1;
	if (g_sched_fn)
		rc = g_sched_fn(g_sched_ctx, b->rot, b->n, nqb, &h->sched);
	if (rc < 0) {
		const uint32_t low = h->tile_bits ? h->low_bits :
			auto_low(h->low_bits);
		/* the cut at tile 13 depends on the half-tile setting; without
		 * that form tile 13 runs one workgroup per CU */
		const uint32_t half = ph2hip_fused_half_mask();
		uint32_t tile = h->tile_bits ? h->tile_bits : auto_tile(nqb);
		if (!h->tile_bits && tile == 13 && !(half >> 13 & 1))
			tile = 12;
		s = &b->sched;
		rc = 0;
		if (!b->scheduled || b->tile != tile ||
		    b->low != h->low_bits ||
		    b->half != half || b->chosen != !h->tile_bits) {
			b->scheduled = 0;
			rc = ph2_sched_greedy(b->rot, b->n, nqb, tile, low,
				&b->sched);
			uint32_t tile2 = tile, low2 = low;
			if (rc == 0 && !h->tile_bits &&
			    second_cut(nqb, h->low_bits, &tile2, &low2) &&
			    (rc = ph2_sched_greedy(b->rot, b->n, nqb, tile2, low2,
				     &h->sched)) == 0 &&
			    take_second(nqb, b->sched.npass, h->sched.npass)) {
				const struct ph2_sched t = b->sched;
				b->sched = h->sched;
				h->sched = t;
			}
			b->tile = tile;
			b->low = h->low_bits;
			b->half = half;
			b->chosen = !h->tile_bits;
			b->scheduled = rc == 0;
		}
	}
	if (rc == 0)
		rc = ph2hip_rotate_fused(h->damp, nqb, b->rot, b->n, s->len,
			s->tile_bits, s->npass, s->low_bits);
	return rc;
}

void qreg_paulirot(struct qreg *reg, struct paulis code_hi,
	const struct paulis *codes_lo, const double *phis, size_t ncodes)
{
	struct qreg_hip *h = reg->backend;
	if (code_hi.pak[0] | code_hi.pak[1]) {
		log_error("qreg_paulirot: hi code on a single-GPU register");
		h->err = -1;
		return;
	}
	if (ncodes == 0)
		return;
	if (settle(h, reg->namp) < 0)
		return;
	struct block *b = block_of(h, codes_lo, phis, ncodes);
	if (!b) {
		log_error("qreg_paulirot: alloc");
		h->err = -1;
		return;
	}
	const uint32_t nqb = reg->qb_lo;
	int rc;
	h->pending |= SENT_WORK;
	if (h->mode == QREG_HIP_PLAIN)
		rc = ph2hip_rotate_plain(h->damp, nqb, b->rot, ncodes);
	else if (nqb < PH2HIP_TILE_MIN)
		rc = ph2hip_rotate_small(h->damp, nqb, b->rot, ncodes);
	else
		rc = rotate_block(h, nqb, b);
	if (rc < 0)
		set_err(reg, "qreg_paulirot");
}
