/*
 * The staged sweep of a half ray (included by mgx_solver.hip, inside its
 * anonymous namespace).
 *
 * A group of 32 lanes takes the quadrature bins of one line on one half ray.
 * What a traced entry contributes besides the bin's frequency -- the line data
 * interpolated at it, its shift, the length of its segment, the branch of the
 * segment and which lines its windows hold -- is the same for every bin, so it
 * is formed once per (line, entry): the lanes of the group take 32 consecutive
 * entries side by side, gather their records from memory together and leave one
 * 80-byte StagedEntry each in LDS.  The bins then walk those entries in order,
 * with two or three broadcast reads from LDS per segment instead of ten
 * dependent gathers, one interpolation (up to three powf per end) per entry
 * instead of one per bin, and no window test where the staging lane has shown
 * its outcome for every bin.
 */

/* what a segment's optical depth needs (seg) and what its inner entry's window holds
   (ent), in StagedEntry::kind */
enum {
    SEG_EMPTY = 0, /* no line in the window of any bin: depth min_opacity dz, no source */
    SEG_SOLO = 1,  /* line-integrated, only the own line in the window of every bin */
    SEG_LANE = 2,  /* line-integrated, each bin tests its window */
    SEG_TRAP = 3,  /* trapezoid rule */
    ENT_EMPTY = 0 << 2,
    ENT_SOLO = 1 << 2,
    ENT_LANE = 2 << 2,
    SEG_MASK = 3,
    ENT_MASK = 3 << 2,
    SEG_IS_TRAP = 1 << 4 /* the trapezoid branch, also when its windows are empty */
};

struct alignas(16) StagedEntry {
    double iw, kap;          /* inverse width and opacity, interpolated */
    double src, eps;         /* emissivity / opacity and emissivity, interpolated */
    double shift, dz;        /* shift; length of the segment from the entry before */
    double fac, ubm;         /* interpolation factor; larger ub of that segment's ends */
    uint32_t nr, nri, kind, pad;
};
static_assert(sizeof(StagedEntry) == 80, "five 16-byte words");

/* Entries a group keeps in LDS: kStage of them are staged together, the last one
   of a chunk again as the first of the next, so that both ends of every segment
   are there. */
constexpr uint32_t kStage = 32;

/* The half ray of a group, in LDS: what staging reads and the sweep does not have to
   hold in registers. */
struct GroupRay {
    uint32_t o, line;
    uint32_t S;               /* steps */
    uint32_t n;               /* entries besides the origin's */
    uint32_t plain;           /* every step is one entry */
    uint32_t list;            /* which of the wave's two walk lists */
    double shift0, shift_c;   /* shift of o: of its step's start, of its own entry */
    double fmin, fmax;        /* smallest and largest bin frequency */
    OwnLine ol;
};

/* a walk list in LDS, and the prefix sums of the group that sweeps it */
struct WalkList {
    const uint32_t *nxt;
    const double *dZ, *sh;
    uint32_t *pre;
};

__device__ __forceinline__ WalkList walk_list(unsigned char *smem, uint32_t cap, uint32_t list, uint32_t grp)
{
    double *dZ = reinterpret_cast<double *>(smem + 8 * ((2 * cap * 4 + 7) / 8));
    WalkList w;
    w.nxt = reinterpret_cast<uint32_t *>(smem) + list * cap;
    w.dZ = dZ + list * cap;
    w.sh = dZ + 2 * cap + list * cap;
    w.pre = reinterpret_cast<uint32_t *>(dZ + 4 * cap) + grp * cap;
    return w;
}

/* sum, smallest and largest over the 32 lanes of a group, in every lane */
template <typename Op>
__device__ __forceinline__ double group32(double v, Op op)
{
    v = op(v, dpp_get<0xb1>(v));
    v = op(v, dpp_get<0x4e>(v));
    v = op(v, dpp_get<0x141>(v));
    v = op(v, dpp_get<0x140>(v));
    double even, odd;
    half_rows(v, even, odd);
    return op(even, odd);
}

/* Interpolation counts of the groups' half rays (o, line, S and list of *g are set):
   pre, n and plain.  ALL takes the largest count over the lines
   (InterpHelper::get_n_interp) instead of the line's own.  All lanes of the wave call
   this together. */
template <bool ALL>
__device__ inline void count_entries(const KParams &kp, unsigned char *smem, GroupRay *g)
{
    const uint32_t q = threadIdx.x & 31;
    const uint32_t grp = (threadIdx.x & (MGX_WAVE - 1)) >> 5;
    const uint32_t S = g->S, o = g->o, line = g->line;
    const WalkList w = walk_list(smem, kp.cap, g->list, grp);
    bool one = true;
    for (uint32_t st = q; st < S; st += 32) {
        const uint32_t crt = (st == 0) ? o : w.nxt[st - 1];
        const uint32_t mm = ALL ? n_interp_all(kp, crt, w.nxt[st])
                                : n_interp_for_line(kp, line, crt, w.nxt[st]);
        if (mm > 0xffffu) atomicOr(&kp.status[0], (uint32_t)ERR_INTERP);
        w.pre[st] = mm > 0xffffu ? 0xffffu : mm;
        one = one && mm == 1;
    }
    const uint64_t many = __ballot(!one);
    uint32_t total = S;
    if (many) {
        __syncthreads();
        total = 0;
        for (uint32_t s0 = 0; s0 < S; s0 += 32) {
            const uint32_t st = s0 + q;
            uint32_t v = st < S ? w.pre[st] : 0;
#pragma unroll
            for (int d = 1; d < 32; d <<= 1) {
                const uint32_t x = __shfl_up(v, d, 32);
                if (q >= (uint32_t)d) v += x;
            }
            if (st < S) w.pre[st] = v + total;
            total += __shfl(v, 31, 32);
        }
    }
    if (q == 0) {
        g->plain = ((many >> (32 * grp)) & 0xffffffffull) == 0;
        g->n = total;
    }
    __syncthreads();
}

/* Which lines the window of every bin holds, for shifts lo <= hi at the two ends
   (equal for an entry): 0 none, 1 the own line alone, 2 each bin has to test.  The
   bins' window edges are left(f) = f lo - W(f) and right(f) = f hi + W(f) with
   W(f) = M (f hi ub); rounding keeps f hi, W and right monotone in f, so the
   values at fmin and fmax bound those of every bin. */
template <int APPROX>
__device__ inline uint32_t group_window(const KParams &kp, const GroupRay &g, double lo, double hi,
                                        double ub)
{
    if (APPROX == MGX_APPROX_ONE_LINE) return 1;
    if (APPROX == MGX_APPROX_NONE) return kp.m.nlines == 1 ? 1 : 2;
    if (!(lo > 0.0)) return 2;
    const double M = kp.op.max_distance_opacity_contribution;
    const double r0 = g.fmin * hi, r1 = g.fmax * hi;
    const double W0 = M * (r0 * ub), W1 = M * (r1 * ub);
    if (!(W0 >= 0.0)) return 2;
    const double left_min = g.fmin * lo - W1, left_max = g.fmax * lo - W0;
    const double right_min = r0 + W0, right_max = r1 + W1;
    if (g.ol.a_lo < left_min && left_max <= g.ol.a_g && g.ol.a_g <= right_min && right_max < g.ol.a_hi)
        return 1;
    if ((g.ol.a_g < left_min && right_max < g.ol.a_hi) || (right_max < g.ol.a_g && g.ol.a_lo < left_min))
        return 0;
    return 2;
}

/* the same for one bin, at the frequencies cf and nf of the two ends */
template <int APPROX>
__device__ __forceinline__ uint32_t lane_window(const KParams &kp, const OwnLine &ol, double cf,
                                                double nf, double ub)
{
    if (APPROX == MGX_APPROX_ONE_LINE) return 1;
    if (APPROX == MGX_APPROX_NONE) return kp.m.nlines == 1 ? 1 : 2;
    const double lf = cf < nf ? cf : nf, rf = cf < nf ? nf : cf;
    const double W = kp.op.max_distance_opacity_contribution * (rf * ub);
    const double left = lf - W, right = rf + W;
    if (!(ol.a_g < left) && ol.a_lo < left && !(right < ol.a_g) && right < ol.a_hi) return 1;
    if ((ol.a_g < left && right < ol.a_hi) || (right < ol.a_g && ol.a_lo < left)) return 0;
    return 2;
}

/* point, partner, factor, shift and segment length (towards the origin) of entry
   number n - q counted from the outer end (q = 0: the origin itself) */
struct EntryGeom {
    Entry e;
    double dz;
};

__device__ inline EntryGeom entry_geom(const GroupRay &g, const WalkList &w, uint32_t s, uint32_t i,
                                       uint32_t m)
{
    EntryGeom r;
    const uint32_t nxt = w.nxt[s], crt = (s == 0) ? g.o : w.nxt[s - 1];
    const double sh_n = w.sh[s], sh_c = (s == 0) ? g.shift0 : w.sh[s - 1];
    r.e.nr = nxt;
    r.e.nri = crt;
    if (m > 1) {
        const double dshift = sh_n - sh_c;
        const double dshift_interpl = dshift / m;
        r.dz = w.dZ[s] / m;
        r.e.ifac = 1.0 - ((double)i) / m;
        r.e.shift = sh_c + i * dshift_interpl;
    } else {
        r.dz = w.dZ[s];
        r.e.ifac = 0.0;
        r.e.shift = sh_n;
    }
    return r;
}

/* Stages entry number k of the group (counted from the outer end, k <= g.n) into *out. */
template <int APPROX, int PREC>
__device__ inline void stage_entry(const KParams &kp, const GroupRay &g, const WalkList &wl, uint32_t k,
                                   StagedEntry *out)
{
    const uint32_t q = g.n - k; /* entries inward of it */
    /* its step s and place i in the step's m entries, and those of the entry outside it */
    uint32_t s = 0, i = 0, m = 1, so = 0, io = 1, mo = 1;
    if (g.plain) {
        s = q - 1; /* unused for the origin (q = 0) */
        i = 1;
        so = q;
    } else {
        uint32_t lo = 0, hi = g.S; /* first step whose entries reach beyond q - 1 */
        while (lo < hi) {
            const uint32_t mid = (lo + hi) / 2;
            if (wl.pre[mid] < q) lo = mid + 1;
            else hi = mid;
        }
        s = lo;
        const uint32_t c = (s > 0) ? wl.pre[s - 1] : 0;
        i = q - c;
        m = wl.pre[s] - c;
        if (q > 0 && i < m) {
            so = s;
            io = i + 1;
            mo = m;
        } else if (k > 0) {
            so = (q == 0) ? 0 : s + 1;
            const uint32_t co = (so > 0) ? wl.pre[so - 1] : 0;
            mo = wl.pre[so] - co;
        }
    }
    EntryGeom me, outer;
    if (q == 0) {
        me.e.nr = me.e.nri = g.o;
        me.e.ifac = 0.0;
        me.e.shift = g.shift_c;
    } else {
        me = entry_geom(g, wl, s, i, m);
    }
    outer = me;
    outer.dz = 0.0;
    if (k > 0) outer = entry_geom(g, wl, so, io, mo);
    const double4 a = lp(kp, me.e.nr, g.line);
    const double2 du = dsm_ub(kp, me.e.nr), du_o = dsm_ub(kp, outer.e.nr);
    StagedEntry r;
    r.iw = a.x;
    r.kap = a.z;
    r.src = a.w;
    r.eps = a.y;
    if (me.e.ifac != 0.0) {
        const double4 b = lp(kp, me.e.nri, g.line);
        r.iw = interp_linear(a.x, b.x, me.e.ifac);
        r.kap = interp_log<PREC>(a.z, b.z, me.e.ifac);
        r.src = interp_log<PREC>(a.w, b.w, me.e.ifac);
        r.eps = interp_log<PREC>(a.y, b.y, me.e.ifac);
    }
    r.shift = me.e.shift;
    r.dz = outer.dz;
    r.fac = me.e.ifac;
    r.ubm = (du.y < du_o.y) ? du_o.y : du.y;
    r.nr = me.e.nr;
    r.nri = me.e.nri;
    r.pad = 0;
    const double dshift_abs = fabs(me.e.shift - outer.e.shift);
    const double dshift_max = (du_o.x < du.x) ? du_o.x : du.x;
    const double lo = me.e.shift < outer.e.shift ? me.e.shift : outer.e.shift;
    const double hi = me.e.shift < outer.e.shift ? outer.e.shift : me.e.shift;
    const uint32_t we = group_window<APPROX>(kp, g, me.e.shift, me.e.shift, du.y);
    const bool floor_ok = kp.op.min_opacity * r.dz > 0.0; /* the depth's lower bound is one */
    uint32_t kind;
    if (dshift_abs > dshift_max) {
        const uint32_t w = group_window<APPROX>(kp, g, lo, hi, r.ubm);
        kind = w == 1 ? SEG_SOLO : (w == 0 && floor_ok) ? SEG_EMPTY : SEG_LANE;
    } else {
        const uint32_t wo = group_window<APPROX>(kp, g, outer.e.shift, outer.e.shift, du_o.y);
        kind = SEG_IS_TRAP | ((we == 0 && wo == 0 && floor_ok) ? SEG_EMPTY : SEG_TRAP);
    }
    r.kind = kind | (we << 2);
    *out = r;
}

/* Stages the entries from number k0 on (count of them, those that exist) of every group
   into its part of the chunk; k0 is the group's own.  All lanes of the wave call this
   together. */
template <int APPROX, int PREC>
__device__ inline void stage_chunk(const KParams &kp, unsigned char *smem, const GroupRay *g, int k0,
                                   uint32_t count, StagedEntry *chunk)
{
    const uint32_t q = threadIdx.x & 31;
    const int k = k0 + (int)q;
    __syncthreads();
    if (g->S > 0 && q < count && k >= 0 && (uint32_t)k <= g->n) {
        const WalkList w = walk_list(smem, kp.cap, g->list, (threadIdx.x & (MGX_WAVE - 1)) >> 5);
        stage_entry<APPROX, PREC>(kp, *g, w, (uint32_t)k, chunk + q);
    }
    __syncthreads();
}

/*
 * Windows that hold several lines.  The lanes of a group take nw (kWindowLines, fewer where
 * LDS is short) lines of the sorted list side by side: those inside the union of the bins'
 * windows have their data gathered and interpolated at the segment's ends (or at one entry) by
 * one lane each and left in LDS, from where every bin adds up the lines of its own window, in
 * order.
 */
constexpr uint32_t kWindowLines = 16;

struct WindowLine {
    double f;                /* line frequency */
    double iw_o, kap_o, src_o; /* outer end; an entry: iw, kap, eps */
    double iw_i, kap_i, src_i; /* inner end */
    uint32_t l, pad;         /* the line */
};

/* line data of line l at a staged entry; EPS: the emissivity in the place of the source */
template <int PREC, bool EPS>
__device__ __forceinline__ void line_at(const KParams &kp, const StagedEntry *e, uint32_t l, double &iw,
                                        double &kap, double &src)
{
    const double4 a = lp(kp, e->nr, l);
    const double t = e->fac;
    iw = a.x;
    kap = a.z;
    src = EPS ? a.y : a.w;
    if (t != 0.0) {
        const double4 b = lp(kp, e->nri, l);
        iw = interp_linear(a.x, b.x, t);
        kap = interp_log<PREC>(a.z, b.z, t);
        src = interp_log<PREC>(EPS ? a.y : a.w, EPS ? b.y : b.w, t);
    }
}

/* optical depth of one line between two ends at frequencies f_o and f_i
   (compute_dtau_single_line, solver.tpp:2374-2455; the ends may be swapped), and its
   derivative dop with respect to the mean opacity */
template <int PREC>
__device__ __forceinline__ double line_depth(double iw_o, double iw_i, double kap_o, double kap_i, double f_o,
                                             double f_i, double linefreq, double dz, double min_opacity,
                                             double &dop)
{
    const double avg_iw = (iw_o + iw_i) / 2.0;
    const double avg_op = (kap_o + kap_i) / 2.0;
    if (f_o == f_i) {
        const double prof = gaussian<PREC>(avg_iw, f_o - linefreq);
        dop = dz * prof;
        return dz * (prof * avg_op + min_opacity);
    }
    const double pos_i = (linefreq - f_i) * avg_iw;
    const double pos_o = (linefreq - f_o) * avg_iw;
    const float erf_diff = mgx_ref_erff((float)pos_i) - mgx_ref_erff((float)pos_o);
    const double h = 0.5 * rcp(pos_i - pos_o);
    const double erfterm = avg_op * (double)erf_diff * h;
    dop = dz * (avg_iw * ((double)erf_diff * h));
    return dz * fma(avg_iw, erfterm, min_opacity);
}

/* sums over a bin's window: ENTRY false: depth, depth x outer source, depth x inner
   source of the segment eo - ei; true: emissivity and opacity of the entry ei */
struct WindowSum {
    double a, b, c;
};

/* the lines at a segment's ends, or at an entry */
template <int PREC, bool ENTRY>
__device__ __forceinline__ void window_line(const KParams &kp, const StagedEntry *eo, const StagedEntry *ei,
                                            double f, uint32_t l, WindowLine &w)
{
    w.f = f;
    line_at<PREC, ENTRY>(kp, ENTRY ? ei : eo, l, w.iw_o, w.kap_o, w.src_o);
    if (ENTRY) {
        w.iw_i = w.kap_i = w.src_i = 0.0;
    } else {
        line_at<PREC, false>(kp, ei, l, w.iw_i, w.kap_i, w.src_i);
    }
    w.l = l;
}

/* a group whose bins' windows lie apart: their union is this many times a bin's own window,
   in a list of more lines than two rounds.  64^2 images of a 7^3 wind, 31 bins over 2.2e-4 of
   a line's frequency, lines 2e-6 apart, all bins together and each by itself: 20 lines 0.72
   and 0.92 ms, 40 lines 1.29 and 1.11, 100 lines 2.60 and 1.16, 300 lines 3.9 and 1.5 (their
   gradients 2.4 and 2.9, 5.1 and 3.6, 13.0 and 3.9, 18.5 and 5.0). */
constexpr double kApart = 4.0;
constexpr uint32_t kApartLines = 2 * kWindowLines;

/* Stages the lines in the windows round by round and hands each to take(line, its index,
   whether it is in the bin's window, whether it is the same for all bins of the group), in the
   sorted order; mine marks the bins that have a window here.  All lanes of the wave call this
   together, and take too.  WIDE: the group's bins need not belong to one line.  Where their
   windows lie apart, most lines of the union are in the windows of a few bins each, and every
   bin takes its own window's lines at the same time instead. */
template <int APPROX, int PREC, bool ENTRY, bool WIDE, typename Take>
__device__ __forceinline__ void window_lines_of(const KParams &kp, const GroupRay *g, WindowLine *lines,
                                                uint32_t nw, const StagedEntry *eo, const StagedEntry *ei,
                                                double f_o, double f_i, bool mine, Take take)
{
    const mgx_model &m = kp.m;
    const uint32_t q = threadIdx.x & 31, grp = (threadIdx.x & (MGX_WAVE - 1)) >> 5;
    const bool any = ((__ballot(mine) >> (32 * grp)) & 0xffffffffull) != 0;
    const double M = kp.op.max_distance_opacity_contribution;
    /* a group without a bin here may stand past its half ray's end: its entries are not
       staged, and their point is not read */
    double ub = ei->ubm;
    if (ENTRY && any) ub = gld(&kp.pts[ei->nr].ub);
    double left = -__builtin_inf(), right = __builtin_inf(); /* the bin's window */
    double left_all = left, right_all = right;               /* the group's */
    if (APPROX == MGX_APPROX_CLOSE_LINES) {
        const double lf = f_o < f_i ? f_o : f_i, rf = f_o < f_i ? f_i : f_o;
        const double W = M * (rf * ub);
        left = lf - W;
        right = rf + W;
        const double s_o = eo->shift, s_i = ei->shift;
        const double lo = s_o < s_i ? s_o : s_i, hi = s_o < s_i ? s_i : s_o;
        if (lo > 0.0) {
            const double r1 = g->fmax * hi;
            const double W1 = M * (r1 * ub);
            left_all = g->fmin * lo - W1;
            right_all = r1 + W1;
        }
    }
    if constexpr (WIDE && APPROX == MGX_APPROX_CLOSE_LINES) {
        if (m.nlines > kApartLines && __ballot(mine && right_all - left_all > kApart * (right - left))) {
            uint32_t s = 0, end = 0;
            if (mine) {
                s = lower_bound_d(m.sorted_line, m.nlines, left);
                end = upper_bound_d(m.sorted_line, m.nlines, right);
            }
#pragma unroll 1
            for (; __ballot(s < end); s++) {
                WindowLine w = {};
                const bool here = s < end;
                if (here)
                    window_line<PREC, ENTRY>(kp, eo, ei, gld(&m.sorted_line[s]), gld(&m.sorted_line_map[s]), w);
                take(&w, w.l, here, false);
            }
            return;
        }
    }
#pragma unroll 1
    for (uint32_t s0 = 0; s0 < m.nlines; s0 += nw) {
        bool in = false;
        double f = 0.0;
        if (any && q < nw && s0 + q < m.nlines) {
            f = APPROX == MGX_APPROX_CLOSE_LINES ? gld(&m.sorted_line[s0 + q]) : gld(&m.line[s0 + q]);
            in = !(f < left_all) && !(right_all < f);
        }
        const uint64_t b = __ballot(in);
        if (b == 0) continue;
        __syncthreads();
        if (in) {
            WindowLine w;
            window_line<PREC, ENTRY>(kp, eo, ei, f,
                                     APPROX == MGX_APPROX_CLOSE_LINES ? gld(&m.sorted_line_map[s0 + q]) : s0 + q, w);
            lines[q] = w;
        }
        __syncthreads();
        /* both groups' lines in turn, so that the lanes of the wave stay together */
        const uint32_t set = (uint32_t)(b >> (32 * grp));
        uint32_t all = (uint32_t)b | (uint32_t)(b >> 32);
        while (all) {
            const uint32_t i = (uint32_t)__ffs((int)all) - 1;
            all &= all - 1;
            const WindowLine *w = lines + i;
            const bool here = mine && ((set >> i) & 1) != 0 && !(w->f < left) && !(right < w->f);
            take(w, w->l, here, true);
        }
    }
    __syncthreads();
}

template <int APPROX, int PREC, bool ENTRY, bool WIDE>
__device__ __forceinline__ WindowSum window_sum(const KParams &kp, const GroupRay *g, WindowLine *lines,
                                                uint32_t nw, const StagedEntry *eo, const StagedEntry *ei,
                                                double f_o, double f_i, bool mine)
{
    WindowSum r = {0.0, ENTRY ? kp.op.min_opacity : 0.0, 0.0};
    window_lines_of<APPROX, PREC, ENTRY, WIDE>(
        kp, g, lines, nw, eo, ei, f_o, f_i, mine, [&](const WindowLine *w, uint32_t, bool in, bool) {
            if (!in) return;
            if (ENTRY) {
                const double prof = gaussian<PREC>(w->iw_o, f_i - w->f);
                r.a += prof * w->src_o;
                r.b += prof * w->kap_o;
            } else {
                double dop;
                const double d = line_depth<PREC>(w->iw_o, w->iw_i, w->kap_o, w->kap_i, f_o, f_i, w->f, ei->dz,
                                                  kp.op.min_opacity, dop);
                r.a += d;
                r.b = fma(d, w->src_o, r.b);
                r.c = fma(d, w->src_i, r.c);
            }
        });
    return r;
}

/* An entry as the next segment's outer end: what a line-integrated segment takes
   from it, held in registers. */
struct OuterEnd {
    double iw, kap, src, f; /* f: the bin's frequency at the entry */
};

/* The bin's own constants of a sweep. */
struct BinLine {
    double freq, a_g; /* the bin's and its own line's frequency */
};

/* emissivity, opacity and own profile value of an entry at a bin's frequency; phi is
   NaN where several lines contribute, 0 where none does.  All lanes of the wave call
   this together; those that want a value pass need. */
template <int APPROX, int PREC, bool WIDE>
__device__ __forceinline__ void staged_eta_chi(const KParams &kp, const GroupRay *g, WindowLine *lines, uint32_t nw,
                                               const BinLine &bin, const StagedEntry *e, bool need,
                                               double &eta, double &chi, double &phi)
{
    const double f = bin.freq * e->shift;
    uint32_t w = need ? (e->kind & ENT_MASK) >> 2 : 0;
    if (w == 2) w = lane_window<APPROX>(kp, g->ol, f, f, gld(&kp.pts[e->nr].ub));
    if (need) {
        phi = 0.0;
        eta = 0.0;
        chi = kp.op.min_opacity;
    }
    if (w == 1) {
        phi = gaussian<PREC>(e->iw, f - bin.a_g);
        eta = 0.0 + phi * e->eps;
        chi = kp.op.min_opacity + phi * e->kap;
    }
    if (__ballot(w == 2)) {
        const WindowSum s = window_sum<APPROX, PREC, true, WIDE>(kp, g, lines, nw, e, e, f, f, w == 2);
        if (w == 2) {
            eta = s.a;
            chi = s.b;
            phi = __builtin_nan("");
        }
    }
}

/*
 * The segment between the staged entries eo and ei at one bin (compute_source_dtau,
 * solver.tpp:2140-2186).  Its value does not depend on which end is the current one.
 * ec_out / ec_in cache the ends' emissivity and opacity (ec_out from the segment
 * before, when that took the trapezoid rule too).  All lanes of the wave call this
 * together; those without a segment pass on = false.  For the adjoint's tape (the other
 * sweeps drop them): raw is the depth before a line-integrated one is clamped, dop
 * d depth / d mean opacity of a segment with the own line alone.
 */
template <int APPROX, int PREC, bool WIDE>
__device__ __forceinline__ void staged_segment(const KParams &kp, const GroupRay *g, WindowLine *lines, uint32_t nw,
                                               const BinLine &bin, const StagedEntry *eo,
                                               const StagedEntry *ei, bool on, OuterEnd &out, PointEC &ec_out,
                                               PointEC &ec_in, double &dtau, double &S_out, double &S_in,
                                               double &raw, double &dop)
{
    const uint32_t kind = ei->kind;
    const double dz = ei->dz;
    OuterEnd in;
    in.iw = ei->iw;
    in.kap = ei->kap;
    in.src = ei->src;
    in.f = bin.freq * ei->shift;
    const double bound = kp.op.min_opacity * dz;
    uint32_t seg = on ? kind & SEG_MASK : SEG_EMPTY;
    dtau = raw = bound;
    dop = S_out = S_in = 0.0;
    if (seg == SEG_LANE) {
        const uint32_t w = lane_window<APPROX>(kp, g->ol, out.f, in.f, ei->ubm);
        seg = w == 1 ? SEG_SOLO : (w == 0 && bound > 0.0) ? SEG_EMPTY : SEG_LANE;
    }
    if (seg == SEG_SOLO) {
        const double d = line_depth<PREC>(out.iw, in.iw, out.kap, in.kap, out.f, in.f, bin.a_g, dz,
                                          kp.op.min_opacity, dop);
        S_out = out.src;
        S_in = in.src;
        dtau = raw = d;
        if (APPROX == MGX_APPROX_CLOSE_LINES && -bound < d && d < bound) {
            /* the clamped depth: the sources keep their share of the line's own */
            const double share = d * rcp(bound);
            dtau = bound;
            S_out *= share;
            S_in *= share;
        }
    }
    if (__ballot(seg >= SEG_LANE)) {
        if (__ballot(seg == SEG_LANE)) {
            const WindowSum v = window_sum<APPROX, PREC, false, WIDE>(kp, g, lines, nw, eo, ei, out.f, in.f, seg == SEG_LANE);
            if (seg == SEG_LANE) {
                double d = raw = v.a;
                if (APPROX == MGX_APPROX_CLOSE_LINES && -bound < d) d = (bound < d) ? d : bound;
                const double rd = rcp(d);
                dtau = d;
                S_out = v.b * rd;
                S_in = v.c * rd;
            }
        }
        double phi;
        const bool trap = seg == SEG_TRAP;
        staged_eta_chi<APPROX, PREC, WIDE>(kp, g, lines, nw, bin, eo, trap && !ec_out.valid, ec_out.eta, ec_out.chi, phi);
        staged_eta_chi<APPROX, PREC, WIDE>(kp, g, lines, nw, bin, ei, trap, ec_in.eta, ec_in.chi, phi);
        if (trap) {
            ec_in.valid = true;
            S_out = ec_out.eta * rcp(ec_out.chi);
            S_in = ec_in.eta * rcp(ec_in.chi);
            dtau = raw = 0.5 * (ec_out.chi + ec_in.chi) * dz;
        }
    }
    out = in;
}
