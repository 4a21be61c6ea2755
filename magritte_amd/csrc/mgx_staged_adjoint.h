/*
 * The reverse sweep of a half ray over staged entries (included by mgx_solver.hip,
 * inside its anonymous namespace).
 *
 * What a segment depends on -- the line data interpolated at its two entries -- is the
 * same for every bin of the group.  So each bin forms the derivative with respect to an
 * entry's source, emissivity, opacity and inverse width (S, E, K, W), these are summed over
 * the group, and only the sums are taken on to the two points the entry is interpolated
 * between: once per (line, entry), by the lanes of the group side by side, whatever the
 * number of bins.
 *   eps_i = eps_a^(1-t) eps_b^t (the same for kappa and for their quotient, the source),
 *   so d eps_i / d eps_a = (1 - t) eps_i / eps_a, d eps_i / d eps_b = t eps_i / eps_b; iw_i
 *   is linear in t.  An entry at a point (t = 0) has the point's own values: the factor is
 *   one and no emissivity or opacity, which may be zero, is divided by.
 *
 * Before, a bin's reverse of an interpolated segment recomputed its erf and powf terms and
 * added to four points by itself, behind a call, and every walk step summed its points over
 * the group.  Measured, forward and backward: J of the 24^3 wind (16% of the entries
 * interpolated), FP64, 33.6 -> 19.0 ms; (log n, T) gradient of a 128^2 image of a clumpy 24^3
 * wind 4.2 -> 2.5 ms.  Four tape words instead of five, two for the half of the segments that
 * no line reaches; the tape and the reverse's own arithmetic bind what is left.
 */

/* Tape of one half ray: segment k (counted from the outer end) stores Y and X of the row
   at its outer entry and, unless the segment is empty for every bin, its depth (before the
   clamp of a line-integrated one) and d depth / d mean opacity of one with the own line
   alone.  Lanes lie side by side within a word.
   The words are doubles in mixed precision too: the reverse forms u_k - u_{k+1} from Y and
   X, which cancels where u is smooth. */
#define MGX_TAPE_WORDS 4
struct Tape {
    /* bytes of one segment's record (all 64 lanes) */
    static constexpr size_t kRecord = (size_t)MGX_WAVE * 8 * MGX_TAPE_WORDS;
    unsigned char *st; /* the half's records, at the lane's word */
    uint32_t cap;      /* segments that fit */
    __device__ __forceinline__ double *at(uint32_t k, uint32_t c) const
    {
        return reinterpret_cast<double *>(st + kRecord * k + (size_t)MGX_WAVE * 8 * c);
    }
};

/* sums of a group's bins for one line at a staged entry: the derivatives with respect to
   its source (of line-integrated segments), emissivity and opacity there, and inverse width */
struct EntryGrad {
    double S, E, K, W;
};

/* where the gradients go; g_iw only in the IW instantiations */
struct GradOut {
    double *eps, *kap, *iw;
};

__device__ __forceinline__ void grad_add(double *g, size_t i, double v)
{
    if (v != 0.0) unsafeAtomicAdd(&g[i], v);
}

/* takes the sums of line l at an entry, whose emissivity, opacity and source are eps, kap
   and src (read where s has a derivative of them), on to its point and partner */
template <bool IW>
__device__ inline void entry_scatter(const KParams &kp, const GradOut &out, const StagedEntry *e, uint32_t l,
                                     double eps, double kap, double src, const EntryGrad &s)
{
    const size_t L = kp.m.nlines, ia = (size_t)e->nr * L + l;
    const double t = e->fac;
    const double4 a = lp(kp, e->nr, l);
    if (IW) grad_add(out.iw, ia, (1.0 - t) * s.W);
    if (t == 0.0) {
        double de = s.E, dk = s.K;
        if (s.S != 0.0) {
            const double r = s.S / a.z;
            de += r;
            dk -= r * a.w;
        }
        grad_add(out.eps, ia, de);
        grad_add(out.kap, ia, dk);
        return;
    }
    /* derivatives with respect to the logarithms */
    const double Ss = s.S != 0.0 ? s.S * src : 0.0;
    const double E = Ss + s.E * eps, K = s.K * kap - Ss;
    const double ta = (t == 1.0) ? 0.0 : 1.0 - t;
    grad_add(out.eps, ia, ta * E / a.y);
    grad_add(out.kap, ia, ta * K / a.z);
    const size_t ib = (size_t)e->nri * L + l;
    const double4 b = lp(kp, e->nri, l);
    grad_add(out.eps, ib, t * E / b.y);
    grad_add(out.kap, ib, t * K / b.z);
    if (IW) grad_add(out.iw, ib, t * s.W);
}

__device__ __forceinline__ double group_sum(double v)
{
    return group32(v, [](double a, double b) { return a + b; });
}

/* the sums over the group, and whether any bin adds something (the same in its lanes) */
template <bool IW>
__device__ __forceinline__ bool group_total(EntryGrad &s)
{
    const uint32_t grp = (threadIdx.x & (MGX_WAVE - 1)) >> 5;
    const uint64_t b_S = __ballot(s.S != 0.0), b_E = __ballot(s.E != 0.0), b_K = __ballot(s.K != 0.0);
    const uint64_t b_W = IW ? __ballot(s.W != 0.0) : 0, b = b_S | b_E | b_K | b_W;
    if (b == 0) return false;
    if (b_S) s.S = group_sum(s.S);
    if (b_E) s.E = group_sum(s.E);
    if (b_K) s.K = group_sum(s.K);
    if (IW) s.W = group_sum(s.W);
    return ((b >> (32 * grp)) & 0xffffffffull) != 0;
}

/* d(gaussian(w, diff))/dw = exp(-x^2) (1 - 2 x^2) / sqrt(pi), x = w diff: the
   derivative of the smooth profile, in double */
__device__ inline double gaussian_dw(double w, double diff)
{
    const double x = w * diff;
    return MGX_INVERSE_SQRT_PI * exp(-x * x) * (1.0 - 2.0 * x * x);
}

/* d(compute_dtau_single_line)/d(avg_iw) at fixed frequencies, of the smooth
   function: dz avg_op d(profile)/dw when the two frequencies are equal, else the
   derivative of dz avg_op (erf(np) - erf(cp)) / (2 (cf - nf)), np = (lf - nf) w,
   cp = (lf - cf) w: dz avg_op (np exp(-np^2) - cp exp(-cp^2)) / (sqrt(pi) (np - cp)) */
__device__ inline double dtau_line_dw(double avg_iw, double avg_op, double linefreq, double cf,
                                      double nf, double dz)
{
    if (cf == nf) return dz * avg_op * gaussian_dw(avg_iw, cf - linefreq);
    const double np = (linefreq - nf) * avg_iw, cp = (linefreq - cf) * avg_iw;
    return dz * avg_op * MGX_INVERSE_SQRT_PI * (np * exp(-np * np) - cp * exp(-cp * cp)) /
           (np - cp);
}

/* Adjoint of one line's part of a line-integrated segment: ld_bar of its depth, so / si
   of its sources at the two ends; dop = d depth / d mean opacity.  Adds to the ends' sums. */
template <bool IW>
__device__ __forceinline__ void line_bwd(const WindowLine &w, double f_o, double f_i, double dz, double dop,
                                         double ld_bar, double so, double si, EntryGrad &o, EntryGrad &i)
{
    const double op_bar = 0.5 * dop * ld_bar;
    o.S += so;
    o.K += op_bar;
    i.S += si;
    i.K += op_bar;
    if (IW && ld_bar != 0.0) {
        const double wb = 0.5 * ld_bar * dtau_line_dw((w.iw_o + w.iw_i) / 2.0, (w.kap_o + w.kap_i) / 2.0, w.f,
                                                      f_o, f_i, dz);
        o.W += wb;
        i.W += wb;
    }
}

/* whether a line-integrated depth is raised to the smallest one, as the forward sweep does */
template <int APPROX>
__device__ __forceinline__ bool depth_clamped(double raw, double bound)
{
    return APPROX == MGX_APPROX_CLOSE_LINES && -bound < raw && raw < bound;
}

/*
 * Reverse of window_sum: the lines of the bins' windows, as window_lines_of hands them
 * on.  ENTRY false: the segment eo - ei with adjoints a_bar of its depth and
 * b_bar, c_bar of its outer and inner source, and the window's sums v (depth unclamped);
 * ENTRY true: the entry ei with adjoints a_bar, b_bar of emissivity and opacity.
 */
template <int APPROX, int PREC, bool ENTRY, bool IW, bool WIDE>
__device__ __forceinline__ void window_bwd(const KParams &kp, const GroupRay *g, WindowLine *lines, uint32_t nw,
                                           const StagedEntry *eo, const StagedEntry *ei, double f_o, double f_i,
                                           bool mine, const WindowSum &v, double a_bar, double b_bar,
                                           double c_bar, const GradOut &out)
{
    const uint32_t q = threadIdx.x & 31;
    /* the adjoints of the sums */
    double sa = a_bar, sb = b_bar, sc = c_bar;
    if (!ENTRY) {
        double d = v.a;
        const double bound = kp.op.min_opacity * ei->dz;
        const bool clamped = depth_clamped<APPROX>(d, bound);
        if (clamped) d = bound;
        const double rd = rcp(d);
        sb = b_bar * rd;
        sc = c_bar * rd;
        sa = clamped ? 0.0 : a_bar - sb * (v.b * rd) - sc * (v.c * rd);
    }
    window_lines_of<APPROX, PREC, ENTRY, WIDE>(
        kp, g, lines, nw, eo, ei, f_o, f_i, mine, [&](const WindowLine *w, uint32_t l, bool in, bool shared) {
            EntryGrad o = {0.0, 0.0, 0.0, 0.0}, i = {0.0, 0.0, 0.0, 0.0};
            if (in && ENTRY) {
                const double prof = gaussian<PREC>(w->iw_o, f_i - w->f);
                i.E = sa * prof;
                i.K = sb * prof;
                if (IW) i.W = gaussian_dw(w->iw_o, f_i - w->f) * (sa * w->src_o + sb * w->kap_o);
            } else if (in) {
                double dop;
                const double d = line_depth<PREC>(w->iw_o, w->iw_i, w->kap_o, w->kap_i, f_o, f_i, w->f, ei->dz,
                                                  kp.op.min_opacity, dop);
                line_bwd<IW>(*w, f_o, f_i, ei->dz, dop, sa + sb * w->src_o + sc * w->src_i, sb * d, sc * d, o, i);
            }
            /* a line that the bins share goes to the points once, a bin's own by itself */
            bool any_o = !ENTRY && in, any_i = in;
            if (shared) {
                any_o = !ENTRY && group_total<IW>(o) && q == 0;
                any_i = group_total<IW>(i) && q == 0;
            }
            if (any_o) entry_scatter<IW>(kp, out, eo, l, 0.0, w->kap_o, w->src_o, o);
            if (any_i) {
                if (ENTRY) /* src_o is the emissivity */
                    entry_scatter<IW>(kp, out, ei, l, w->src_o, w->kap_o, 0.0, i);
                else
                    entry_scatter<IW>(kp, out, ei, l, 0.0, w->kap_i, w->src_i, i);
            }
        });
}

/* derivatives of a row  u + A_a (u - u_a) + A_b (u - u_b) = S  with respect to d_a and d_b,
   A_a = 2/((d_a + d_b) d_a), A_b = 2/((d_a + d_b) d_b); Da = u - u_a, Db = u - u_b */
__device__ inline double2 row_dd(double da, double db, double Da, double Db)
{
    const double rs = rcp(da + db), ra = rcp(da), rb = rcp(db);
    const double Aa = 2.0 * rs * ra, Ab = 2.0 * rs * rb;
    double2 r;
    r.x = -Aa * (rs + ra) * Da - Ab * rs * Db;
    r.y = -Ab * (rs + rb) * Db - Aa * rs * Da;
    return r;
}

/* derivative of a boundary row  (1 + 2/d) u + (2/d^2)(u - u_n) = S + 2 I/d  w.r.t. d */
__device__ inline double bdy_row_dd(double d, double I, double u, double Dn)
{
    const double r = rcp(d);
    return 2.0 * r * r * (I - u) - 4.0 * r * r * r * Dn;
}

/*
 * Reverse pass over one half ray, outward from the centre.  With the system
 * T u = r of the ray (rows as in the reference's elimination) and the seed
 * ubar at the centre, lam = T^-T e_c ubar = D T^-1 D^-1 e_c ubar (D T is
 * symmetric, D = half the sum of a row's two segment depths, or half the one
 * depth of a boundary row), so lam_k = D_k mu_k with mu_k = XI_k mu_{k+1}, the
 * same factors that give u_k = Y_k + XI_k u_{k+1}.  dL/dS_k = lam_k and
 * dL/dd = -sum_rows lam_row dR_row/dd; the differences u_k - u_{k+1} are taken
 * as Y_k - X_k XI_k u_{k+1} (optically thin steps leave u constant to ~13
 * digits, so subtracting two u values would lose them).
 *
 * Segment sources as the reference uses them (row n takes Scurr of segment n,
 * the last row Snext of the last segment): rr-side half (backward = false):
 * a segment supplies its outer row, and its inner source feeds the centre row when
 * the centre is the last row; antipod-side half: a segment supplies the row of
 * its inner entry and the outermost one the boundary row.
 */
struct RevCentre {
    double u, mu, lam; /* u, D^-1-scaled adjoint and adjoint of the centre row */
    double dbar;       /* the centre row's part of dL/d(depth of the innermost segment) */
    bool centre_last;  /* rr-side half only: the centre is the system's last row */
};

/* adjoints an entry collects: of its own line's values, and of emissivity and opacity
   from the trapezoid segments on either side (values in eta, chi) */
struct EntryBar {
    EntryGrad s;
    double eta, chi, phi, eta_bar, chi_bar;
    bool have;
};

template <int APPROX, int PREC, bool IW, bool WIDE>
__device__ __forceinline__ void reverse_half(const KParams &kp, unsigned char *smem, const GroupRay *g,
                                             bool backward, double freq, bool active, StagedEntry *chunk,
                                             EntryGrad *sums, const Tape &tape, double I_b,
                                             const RevCentre &rc, const GradOut &out)
{
    const uint32_t count = kp.stage, q = threadIdx.x & 31;
    const uint32_t n_all = g->n, n = active ? n_all : 0;
    const uint32_t nA = (uint32_t)__builtin_amdgcn_readlane((int)n_all, 0);
    const uint32_t nB = (uint32_t)__builtin_amdgcn_readlane((int)n_all, 32);
    const uint32_t nmax = nA > nB ? nA : nB;
    const BinLine bin = {freq, g->ol.a_g};
    const uint32_t nw = window_lines(count);
    WindowLine *lines = reinterpret_cast<WindowLine *>(smem + lines_lds_offset(kp.cap, count)) +
                        ((threadIdx.x & (MGX_WAVE - 1)) >> 5) * nw;
    double u_in = rc.u, mu_in = rc.mu, lam_in = rc.lam, dbar = rc.dbar;
    EntryBar in = {{0.0, 0.0, 0.0, 0.0}, 0.0, 0.0, 0.0, 0.0, 0.0, false};
    double Y = 0.0, X = 0.0, XI = 0.0, raw = 0.0, gk = 0.0;
    bool first = true;
    for (uint32_t done = 0; done < nmax; done += count - 1) {
        /* entries k0 .. k0 + count - 1 of each group; the innermost one left is the last */
        const int k0 = (int)n_all - (int)done - (int)(count - 1);
        stage_chunk<APPROX, PREC>(kp, smem, g, k0, count, chunk);
        if (q < count) sums[q] = EntryGrad{0.0, 0.0, 0.0, 0.0};
        __syncthreads();
        const uint32_t left = nmax - done, jmin = left < count - 1 ? count - left : 1;
        for (uint32_t j = count - 1; j >= jmin; j--) {
            const int k = k0 + (int)j; /* segment between entries k - 1 and k */
            const bool on = k >= 1 && n > 0;
            const StagedEntry *eo = chunk + j - 1, *ei = chunk + j;
            const double dz = ei->dz, bound = kp.op.min_opacity * dz, bound_n = kp.op.min_opacity * eo->dz;
            const uint32_t kind = on ? ei->kind : (uint32_t)SEG_EMPTY;
            uint32_t seg = kind & SEG_MASK;
            const uint32_t seg_n = on && k >= 2 ? eo->kind & SEG_MASK : (uint32_t)SEG_EMPTY;
            const double f_i = freq * ei->shift, f_o = freq * eo->shift;
            double Yn = 0.0, Xn = 0.0, XIn = 0.0, raw_n = 0.0, gn = 0.0;
            double u_k = 0.0, mu_k = 0.0, lam_k = 0.0, dbar_next = 0.0;
            if (on) {
                if (first) {
                    Y = *tape.at(k - 1, 0);
                    X = *tape.at(k - 1, 1);
                    XI = rcp(1.0 + X);
                    raw = bound;
                    if (seg != SEG_EMPTY) {
                        raw = *tape.at(k - 1, 2);
                        gk = *tape.at(k - 1, 3);
                    }
                    first = false;
                }
                if (k >= 2) {
                    Yn = *tape.at(k - 2, 0);
                    Xn = *tape.at(k - 2, 1);
                    raw_n = bound_n;
                    if (seg_n != SEG_EMPTY) {
                        raw_n = *tape.at(k - 2, 2);
                        gn = *tape.at(k - 2, 3);
                    }
                }
                const double d = seg != SEG_TRAP && depth_clamped<APPROX>(raw, bound) ? bound : raw;
                u_k = fma(XI, u_in, Y);
                mu_k = XI * mu_in;
                const double Din = fma(-X * XI, u_in, Y); /* u_k - u_in */
                if (k >= 2) {
                    const double dn = seg_n != SEG_TRAP && depth_clamped<APPROX>(raw_n, bound_n) ? bound_n : raw_n;
                    lam_k = 0.5 * (dn + d) * mu_k;
                    XIn = rcp(1.0 + Xn);
                    if (seg != SEG_EMPTY || seg_n != SEG_EMPTY) {
                        /* u_k - u_{k-1} = X_{k-1} XI_{k-1} u_k - Y_{k-1} */
                        const double Dout = fma(Xn * XIn, u_k, -Yn);
                        const double2 r = row_dd(d, dn, Din, Dout);
                        dbar -= lam_k * r.x;
                        dbar_next = -lam_k * r.y;
                    }
                } else {
                    lam_k = 0.5 * d * mu_k;
                    if (seg != SEG_EMPTY) dbar -= lam_k * bdy_row_dd(d, I_b, u_k, Din);
                }
            }
            EntryBar eb = {{0.0, 0.0, 0.0, 0.0}, 0.0, 0.0, 0.0, 0.0, 0.0, false}; /* the outer entry */
            const double so = backward ? (k == 1 ? lam_k : 0.0) : lam_k;
            const double si = backward ? lam_in : (k == (int)n && rc.centre_last ? rc.lam : 0.0);
            if (seg == SEG_LANE) {
                const uint32_t w = lane_window<APPROX>(kp, g->ol, f_o, f_i, ei->ubm);
                seg = w == 1 ? SEG_SOLO : (w == 0 && bound > 0.0) ? SEG_EMPTY : SEG_LANE;
            }
            if (seg == SEG_SOLO) {
                /* one line: unclamped, the segment's sources are the line's own and the adjoint
                   of its depth is dbar (the source terms cancel exactly); clamped, the depth is
                   the bound and the sources scale with the line's */
                const WindowLine w = {bin.a_g, eo->iw, eo->kap, eo->src, ei->iw, ei->kap, ei->src, 0u, 0u};
                double ld_bar = dbar, a = so, b = si;
                if (depth_clamped<APPROX>(raw, bound)) {
                    const double rb = rcp(bound), share = raw * rb;
                    ld_bar = (so * w.src_o + si * w.src_i) * rb;
                    a *= share;
                    b *= share;
                }
                line_bwd<IW>(w, f_o, f_i, dz, gk, ld_bar, a, b, eb.s, in.s);
            }
            if (__ballot(seg >= SEG_LANE)) {
                const bool gen = seg == SEG_LANE, trap = seg == SEG_TRAP;
                if (__ballot(gen)) {
                    const WindowSum v = window_sum<APPROX, PREC, false, WIDE>(kp, g, lines, nw, eo, ei, f_o, f_i, gen);
                    window_bwd<APPROX, PREC, false, IW, WIDE>(kp, g, lines, nw, eo, ei, f_o, f_i, gen, v, dbar, so, si,
                                                        out);
                }
                staged_eta_chi<APPROX, PREC, WIDE>(kp, g, lines, nw, bin, eo, trap, eb.eta, eb.chi, eb.phi);
                staged_eta_chi<APPROX, PREC, WIDE>(kp, g, lines, nw, bin, ei, trap && !in.have, in.eta, in.chi, in.phi);
                if (trap) {
                    eb.have = in.have = true;
                    const double ro = rcp(eb.chi), ri = rcp(in.chi);
                    eb.chi_bar += 0.5 * dz * dbar - so * eb.eta * ro * ro;
                    in.chi_bar += 0.5 * dz * dbar - si * in.eta * ri * ri;
                    eb.eta_bar += so * ro;
                    in.eta_bar += si * ri;
                }
            }
            /* the inner entry has all its contributions now, and so has the outermost one */
            const auto finish = [&](EntryBar &e, const StagedEntry *se, EntryGrad *sum, bool here) {
                const bool own = here && e.have && e.phi == e.phi;
                const bool multi = here && e.have && !(e.phi == e.phi) && (e.eta_bar != 0.0 || e.chi_bar != 0.0);
                if (own) {
                    /* eta = phi eps, chi = chi_min + phi kappa */
                    e.s.E += e.eta_bar * e.phi;
                    e.s.K += e.chi_bar * e.phi;
                    if (IW && e.phi != 0.0)
                        e.s.W += gaussian_dw(se->iw, freq * se->shift - bin.a_g) *
                                 (se->eps * e.eta_bar + se->kap * e.chi_bar);
                }
                if (__ballot(multi)) {
                    const double f = freq * se->shift;
                    const WindowSum none = {0.0, 0.0, 0.0};
                    window_bwd<APPROX, PREC, true, IW, WIDE>(kp, g, lines, nw, se, se, f, f, multi, none, e.eta_bar,
                                                       e.chi_bar, 0.0, out);
                }
                EntryGrad t = here ? e.s : EntryGrad{0.0, 0.0, 0.0, 0.0};
                if (group_total<IW>(t) && q == 0) *sum = t;
            };
            finish(in, ei, &sums[j], on);
            if (__ballot(on && k == 1)) finish(eb, eo, &sums[j - 1], on && k == 1);
            if (on) {
                in = eb;
                u_in = u_k;
                mu_in = mu_k;
                lam_in = lam_k;
                dbar = dbar_next;
                Y = Yn;
                X = Xn;
                XI = XIn;
                raw = raw_n;
                gk = gn;
            }
        }
        /* the chunk's sums go to the points; its first entry comes again, unless it is the
           outermost one */
        __syncthreads();
        const int ks = k0 + (int)q;
        if (q < count && ks >= 0 && (q > 0 || ks == 0) && ks <= (int)n_all) {
            const EntryGrad t = sums[q];
            const StagedEntry *se = chunk + q;
            if (t.S != 0.0 || t.E != 0.0 || t.K != 0.0 || (IW && t.W != 0.0))
                entry_scatter<IW>(kp, out, se, g->line, se->eps, se->kap, se->src, t);
        }
        __syncthreads();
    }
}
