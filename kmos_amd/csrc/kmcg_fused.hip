// kmcg_fused.hip -- the fused step loop of single-layer local_smart models.
//
// Included by kmcg_engine.hip (device part, inside its namespace).
//
// A process that runs has every one of its conditions fulfilled (its lists
// match the lattice), so the species of all its condition sites are known
// before any lattice read, before and after each of its writes.  The
// library therefore folds the put/take routines of one process into ONE
// flat list of list updates (build_fused in kmcg_engine.hip): updates whose
// conditions contradict the known species are gone, conditions the known
// species fulfil are dropped, and what is left reads only sites the process
// does not write -- ZGB keeps 15 updates per process with at most one
// condition each (generic: 17 with two), RuO2 38 with one (45 with two).
// Every update is one lane's work; the updates of one process are
// neighbouring lanes, in the reference's order, so the lane that owns the
// process finds its entries as a run of bits of one ballot and fetches them
// with ds_bpermute: no mailboxes, no LDS atomics, no rounds.
//
// What bounds a step is its chain of dependent latencies: the read of the
// picked site, the evaluation, the list reads, the selection of the next
// process.  Deletions are of registered entries only (their conditions
// hold), so the counts after the step are known from the ballots alone; the
// next step is selected from them and ITS site read issued before the list
// updates of this step run.  A slot the updates overwrite is patched in a
// register.  One HBM round trip per step stays on the chain.
//
// Measured against the generic loop: RuO2, one 64x64 trajectory, 3.83 ->
// 2.19 us per step; per 1000 steps ZGB 4096 x 128x128 5.42 -> 3.33 ms, the
// RuO2 mix of 2048 5.38 -> 3.66 ms; tracking on the pairwise model (264
// updates in five chunks) 14.2 -> 10.3 us per step.
//
// Record of one lane (RW words; all chunks of a process in turn):
//   word 0: process - 1 (6 bits) | deletes << 6 | valid << 7
//           | first lane << 8 | lanes << 16 of the updates of process
//           (lane + 1) | conditions << 24 | chunks of this process << 27
//   word 1: the update's site
//   words 2.. : conditions, site and species code
//   last word: a lattice write, site | old << 26 | new << 29 (old == new: none)
// site word: dx, dy, dz (7 bits each) | site type - 1 (5 bits) << 21, from
// the cell of the picked site; species code << 26: species + 1 for the
// 2-bit lattice, the species otherwise.

// bits [off, off + w) of v, sign-extended / zero-extended
__device__ __forceinline__ int bf_s(int v, int off, int w) { return __builtin_amdgcn_sbfe(v, off, w); }
__device__ __forceinline__ int bf_u(int v, int off, int w) { return (int)__builtin_amdgcn_ubfe((unsigned)v, off, w); }

// the 0-based site a site word names, from the uniform cell (x, y, z) with
// first site lb; IN: no offset of the program wraps there
template <bool IN>
__device__ __forceinline__ int fz_site(const Dims &d, int lb, int x, int y, int z, int w)
{
    const int dx = bf_s(w, 0, 7), dy = bf_s(w, 7, 7), n1 = bf_u(w, 21, 5);
    if (IN) {
        int s = lb + n1 + __mul24(dx, d.spuck) + __mul24(dy, d.sX);
        if (d.dim >= 3)
            s += __mul24(bf_s(w, 14, 7), d.sXY);
        return s;
    }
    const int xx = wrap1(x + dx, d.X);
    const int yy = d.dim >= 2 ? wrap1(y + dy, d.Y) : 0;
    const int zz = d.dim >= 3 ? wrap1(z + bf_s(w, 14, 7), d.Z) : 0;
    return d.lin(xx, yy, zz) + n1;
}

// a site's species code as the records hold it
template <int BITS>
__device__ __forceinline__ int fz_code(const unsigned char *lat, int s)
{
    if (BITS == 8)
        return (int)lat[s];
    const unsigned w = *(const unsigned *)(lat + (((unsigned)s >> 2) & ~3u));
    return bf_u((int)w, (s << 1) & 31, 2);
}

template <int NC>
struct FzRec {
    static constexpr int RW = NC <= 1 ? 4 : 8;
    int w0, site, cond[NC], wr;
};

template <int NC>
__device__ __forceinline__ void fz_load(const int *recs, int idx, int lane, FzRec<NC> &q)
{
    // uniform record block, one record per lane: 16-byte loads
    const int4 *p = (const int4 *)(recs + (size_t)idx * (64 * FzRec<NC>::RW)) + lane * (FzRec<NC>::RW / 4);
    const int4 a = p[0];
    q.w0 = a.x;
    q.site = a.y;
    q.cond[0] = a.z;
    if (NC <= 1) {
        q.wr = a.w;
    } else {
        const int4 b = p[1];
        q.cond[1 % NC] = a.w;
        q.cond[2 % NC] = b.x;
        q.cond[3 % NC] = b.y;
        q.cond[4 % NC] = b.z;
        q.wr = b.w;
    }
}

// One lane's update: its site and whether its conditions hold, on the
// lattice before the step's writes; ws: the site of the lane's write.
template <int BITS, int NC, bool IN>
__device__ __forceinline__ bool fz_eval(const Wave<1, BITS> &W, const FzRec<NC> &q, int x, int y, int z, int &s1,
                                        int &ws)
{
    const int lb = W.d.lin(x, y, z);
    int cs[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c)
        cs[c] = fz_site<IN>(W.d, lb, x, y, z, q.cond[c]);
    int got[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c)
        got[c] = fz_code<BITS>(W.lat.p, cs[c]);
    s1 = fz_site<IN>(W.d, lb, x, y, z, q.site) + 1;
    ws = fz_site<IN>(W.d, lb, x, y, z, q.wr);
    const int nc = bf_u(q.w0, 24, 3);
    bool ok = (q.w0 & 128) != 0;
#pragma unroll
    for (int c = 0; c < NC; ++c)
        ok = ok && (c >= nc || got[c] == bf_u(q.cond[c], 26, 6));
    return ok;
}

// the list words one owner lane replays a block of up to RB updates with
struct FzList {
    Rows L;
    int V;
    int pk;          // the slot the next step's site is read from (-1: another lane's list)
    int patch;       // its new content when an update of this step writes it
};

// Up to RB entries of this lane's list, in order (add_proc/del_proc,
// base.mpy:211-301); bits / dbits: the remaining entries and which of them
// delete, relative to lane `a`; s1 and bv0 are the update lanes' sites and
// back-indices, tv[j] the list slot nr - j.  As in replay_block a window of
// slots [nr0-RB+1, nr0+RB] and the back-indices the block itself changes
// stay at hand: in registers for one or two entries (no LDS round trip per
// entry), in LDS for four.  Every lane takes part.
template <int RB, int BITS>
__device__ __forceinline__ void fz_replay(const Wave<1, BITS> &W, FzList &F, int &nr, unsigned &bits, unsigned dbits,
                                          int a, int s1, int bv0, const int (&tv)[RB], int &err)
{
    int st[RB], bv[RB];
    bool act[RB], isdel[RB];
#pragma unroll
    for (int i = 0; i < RB; ++i) {
        act[i] = bits != 0;
        const int rel = act[i] ? __builtin_ctz(bits) : 0;
        const int src = (a + rel) << 2;
        st[i] = __builtin_amdgcn_ds_bpermute(src, s1);
        bv[i] = __builtin_amdgcn_ds_bpermute(src, bv0);
        isdel[i] = act[i] && ((dbits >> rel) & 1);
        bits &= bits - 1;
    }
    const int nr0 = nr;
    const int base = nr0 - (RB - 1);
    int *w = W.win + WIN * W.lane;
    int wr[2 * RB];
#pragma unroll
    for (int j = 0; j < RB; ++j) {
        if (RB > 2)
            w[RB - 1 - j] = tv[j];
        else
            wr[RB - 1 - j] = tv[j];
        wr[RB + j] = 0;
    }
    int cur = nr0;
#pragma unroll
    for (int i = 0; i < RB; ++i) {
        if (RB > 2 && !__ballot(act[i]))
            break;
        if (act[i]) {
            const int site = st[i];
            if (!isdel[i]) {
                if (cur + 1 > F.V) {
                    err |= 2;
                } else {
                    cur += 1;
                    F.L.s(cur) = site;
                    F.L.b(site) = cur;
                    F.patch = cur == F.pk ? site : F.patch;
                    if (RB > 2) {
                        w[cur - base] = site;
                    } else {
#pragma unroll
                        for (int k = 0; k < 2 * RB; ++k)
                            wr[k] = cur - base == k ? site : wr[k];
                    }
#pragma unroll
                    for (int j = i + 1; j < RB; ++j)
                        bv[j] = st[j] == site ? cur : bv[j];
                }
            } else {
                const int mpos = bv[i], last = cur;
                if (mpos == 0) {
                    err |= 2;           // registered by its conditions, not by its list
                } else {
                    if (mpos < last) {
                        int moved = 0;
                        if (RB > 2) {
                            moved = w[last - base];
                        } else {
#pragma unroll
                            for (int k = 0; k < 2 * RB; ++k)
                                moved = last - base == k ? wr[k] : moved;
                        }
                        F.L.s(mpos) = moved;
                        F.L.b(moved) = mpos;
                        F.patch = mpos == F.pk ? moved : F.patch;
                        if (RB > 2) {
                            if (mpos >= base)
                                w[mpos - base] = moved;
                        } else {
#pragma unroll
                            for (int k = 0; k < 2 * RB; ++k)
                                wr[k] = mpos - base == k ? moved : wr[k];
                        }
#pragma unroll
                        for (int j = i + 1; j < RB; ++j)
                            bv[j] = st[j] == moved ? mpos : bv[j];
                    }
                    F.L.s(last) = 0;
                    F.L.b(site) = 0;
#pragma unroll
                    for (int j = i + 1; j < RB; ++j)
                        bv[j] = st[j] == site ? 0 : bv[j];
                    cur = last - 1;
                }
            }
        }
    }
    nr = cur;
}

// do_kmc_steps for one replica per wave (proclist_generic_subroutines.mpy:
// 1-44), fused form.  The launch guarantees: local_smart, one layer, at most
// 64 processes, lists matching the lattices, the lattice in LDS, no extent
// below 2 * fz_moff + 1 (no two offsets of the program meet), NCH chunks of
// 64 records per process (NC <= 1: one).
template <int BITS, int NC, bool MSD>
__device__ __forceinline__ void fused_loop(const KParams &kp, unsigned char *smem)
{
    Wave<1, BITS> W;
    const int r = wave_setup<1, BITS, true, false>(W, kp, smem);
    if (r < 0)
        return;
    const int slot = blockIdx.x * kp.wpg + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = W.lane, P = W.P;
    const int *recs = kp.fz_recs;
    const int nch = NC <= 1 ? 1 : kp.fz_nch;
    const int st0 = kp.status[r];
    long long n = kp.nsteps;
    if (kp.budget)
        n = min(n, kp.budget[slot]);
    if (st0 != ST_OK)
        n = 0;
    if (kp.srec)
        count_species<1, BITS>(W);
    double t = kp.ktime[r], dt_last = kp.kdt[r];
    long long ks = kp.kstep[r];
    unsigned long long ctr = kp.rngctr[r];
    const unsigned seed = kp.seed[r], stream = kp.stream[r];
    int st = st0;
    long long done = 0;
    int rec_left = kp.sample_every;
    long long rec_idx = 0;
    const unsigned row = (unsigned)W.V1 << 2;         // bytes of one list
    FzList F;
    F.L.base = (char *)W.avail;
    F.L.so = row * (unsigned)(lane < P ? lane : 0);
    F.L.bo = row * (unsigned)(P + (lane < P ? lane : 0));
    F.V = W.d.V;
    F.pk = -1;
    F.patch = 0;
    // uniforms of 64 steps at a time, as in steps_loop
    double lmlog = 0.0, lu1 = 0.0, lu2 = 0.0;
    unsigned long long ubase = ctr;
    int uj = 64;
    // the selected step: its terms, total, process, slot, site on the way
    double acc[1] = {0.0};
    double c[1] = {0.0};
    double total = 0.0;
    int pick = 0, kk = 0, sv = 0;
    int nrs = 0;                     // counts the prefixes in acc belong to
    double mlog = 0.0;
    FzRec<NC> q;
    // selects the step after the counts nrx: uniforms, accum_rates, process,
    // slot; its site read and records are issued, not waited for
    auto select = [&](int nrx, bool anew) {
        if (uj == 64) {
            double uu[3];
            step_uniforms(seed, stream, ubase + lane, uu);
            lmlog = -log(uu[0]);
            lu1 = uu[1];
            lu2 = uu[2];
            ubase += 64;
            uj = 0;
        }
        c[0] = (double)nrx * W.rate[0];
        const unsigned long long ch = __ballot(nrx != nrs);
        const int first[1] = {anew ? 0 : ch ? __ffsll((long long)ch) - 1 : 64};
        nrs = nrx;
        total = accumulate<1>(c, acc, P, lane, first);
        if (total > 0.0) {
            pick = interval_search<1>(acc, readlane_d(lu1, uj) * total, P, lane);
            const int nrp = readlane_i(nrx, pick);
            kk = (int)(1.0 + readlane_d(lu2, uj) * (double)nrp);
            kk = __builtin_amdgcn_readfirstlane(kk > nrp ? nrp : kk);
            F.pk = lane == pick ? kk : -1;
            F.patch = 0;
            sv = *(const int *)(F.L.base + (row * (unsigned)pick + ((unsigned)max(kk, 0) << 2)));
            fz_load<NC>(recs, pick * nch, lane, q);
        }
        mlog = readlane_d(lmlog, uj);
        uj += 1;
    };
    if (n > 0)
        select(W.nr[0], true);
#if KMCG_PHASES
    for (int i = 0; i < 5; ++i)
        W.tph[i] = 0;
    W.nblk = W.napply = 0;
    W.tmark = __builtin_amdgcn_s_memtime();
#endif
    while (done < n) {
        if (!(total > 0.0)) {
            st = ST_ABSORBING;
            break;
        }
        PH_MARK(W, 4);
        // this step's site: read ahead, or just written by the last step
        const int pv = readlane_i(F.patch, pick);
        const int site = pv ? pv : __builtin_amdgcn_readfirstlane(sv);
        PH_MARK(W, 1);
        const int cpick = pick;
        const double ctotal = total, cc = c[0], cmlog = mlog;
        if (kk < 1) {                       // only a corrupted database gets here
            st = ST_CORRUPT;
            ctr += 1;
            dt_last = cmlog / ctotal;
            t = t + dt_last;
            ks += 1;
            W.integ[0] = W.integ[0] + cc * dt_last;
            break;
        }
        const int s0 = site - 1;
        const int cell = divm(s0, W.ms);
        const int yz = divm(cell, W.mx);
        const int x = cell - yz * W.d.X;
        const int z = divm(yz, W.my);
        const int y = yz - z * W.d.Y;
        const bool inside = W.d.interior(x, y, z);
        int err = 0;
        const int nchp = NC <= 1 ? 1 : __builtin_amdgcn_readfirstlane(bf_u(q.w0, 27, 5));
        for (int ci = 0; ci < nchp; ++ci) {
            int s1, ws;
            bool ok;
            if (inside)
                ok = fz_eval<BITS, NC, true>(W, q, x, y, z, s1, ws);
            else
                ok = fz_eval<BITS, NC, false>(W, q, x, y, z, s1, ws);
            const bool del = (q.w0 & 64) != 0;
            const unsigned long long mk = __ballot(ok), dk = __ballot(ok && del);
            // back[site] of a deletion
            const unsigned bo = (__umul24((unsigned)W.V1, P + (q.w0 & 63)) + (unsigned)s1) * 4u;
            int bv = 0;
            if (ok && del)
                bv = *(const int *)(F.L.base + bo);
            // the owner lane's entries: a run of the update lanes
            const int a = bf_u(q.w0, 8, 6), len = bf_u(q.w0, 16, 6);
            unsigned bits = (unsigned)bf_u((int)(mk >> a), 0, len);
            const unsigned dbits = (unsigned)bf_u((int)(dk >> a), 0, len);
            const int ne = __popc(bits), nd = __popc(dbits);
            const int nrx = W.nr[0] + ne - 2 * nd;
            int tv[RBLK];
            tv[0] = nd > 0 ? F.L.s(W.nr[0]) : 0;
            tv[1] = tv[2] = tv[3] = 0;
            const bool two = __ballot(ne > 1), four = __ballot(ne > 2);
            if (two)
                tv[1] = nd > 1 ? F.L.s(max(W.nr[0] - 1, 0)) : 0;
            if (four) {
                tv[2] = nd > 2 ? F.L.s(max(W.nr[0] - 2, 0)) : 0;
                tv[3] = nd > 3 ? F.L.s(max(W.nr[0] - 3, 0)) : 0;
            }
            const int wrw = q.wr;
            const bool lastc = ci == nchp - 1;
            PH_MARK(W, 2);
            if (lastc)
                select(nrx, false);
            else
                fz_load<NC>(recs, cpick * nch + ci + 1, lane, q);
            PH_MARK(W, 0);
            // the writes (their old species are known); nothing of this
            // step reads a written site
            if (((unsigned)wrw >> 29) != ((unsigned)(wrw >> 26) & 7u)) {
                const int o = (wrw >> 26) & 7, v = (int)((unsigned)wrw >> 29);
                W.lat.xset(ws, o, v);
                if (W.track) {
                    const int tt = bf_u(wrw, 21, 5);
                    atomicAdd(&W.occ[o * W.d.spuck + tt], -1);
                    atomicAdd(&W.occ[v * W.d.spuck + tt], 1);
                }
            }
            wave_sync();
            if (lastc) {
                // update_clocks, update_integ_rate with the counts before
                const double dt = cmlog / ctotal;
                t = t + dt;
                dt_last = dt;
                W.integ[0] = W.integ[0] + cc * dt;
                W.pstat[0] += lane == cpick ? 1 : 0;
                ctr += 1;
                ks += 1;
                done += 1;
                if (MSD) {
                    if (kp.acf_pa)
                        acf_before<1, BITS>(W, kp, r, t, dt, cpick, site);
                    else
                        msd_track<1, BITS>(W, kp, r, cpick, site);
                }
            }
            // the list updates
#if KMCG_PHASES
            W.napply += 1;
            W.nblk += 1;
#endif
            if (four) {
                fz_replay<RBLK, BITS>(W, F, W.nr[0], bits, dbits, a, s1, bv, tv, err);
                while (__ballot(bits != 0)) {
#if KMCG_PHASES
                    W.nblk += 1;
#endif
                    // the next four: their list tail is read now (slots the
                    // block before wrote are in order behind its stores)
                    int tn[RBLK];
#pragma unroll
                    for (int j = 0; j < RBLK; ++j)
                        tn[j] = bits ? F.L.s(max(W.nr[0] - j, 0)) : 0;
                    // back-indices the blocks before changed: read again
                    int bn = 0;
                    if (ok && del)
                        bn = *(const int *)(F.L.base + bo);
                    fz_replay<RBLK, BITS>(W, F, W.nr[0], bits, dbits, a, s1, bn, tn, err);
                }
            } else if (two) {
                const int t2[2] = {tv[0], tv[1]};
                fz_replay<2, BITS>(W, F, W.nr[0], bits, dbits, a, s1, bv, t2, err);
            } else {
                const int t1[1] = {tv[0]};
                fz_replay<1, BITS>(W, F, W.nr[0], bits, dbits, a, s1, bv, t1, err);
            }
            PH_MARK(W, 3);
        }
        if (MSD && kp.acf_pa && lane == 0)
            acf_after(kp, r);
        if (__ballot(err)) {
            st = ST_CORRUPT;
            break;
        }
        if (W.track && --rec_left == 0) {
            write_record<1, BITS>(W, kp, slot, rec_idx, t, dt_last, ks, ST_OK);
            rec_left = kp.sample_every;
            rec_idx += 1;
        }
    }
    steps_end<1, BITS, true>(W, kp, r, slot, t, dt_last, ks, ctr, st, done);
}

template <int BITS, int NC, bool MSD>
__global__ __launch_bounds__(64 * MAX_WPG) __attribute__((amdgpu_waves_per_eu(4))) void kmc_steps_kernel_fz(KParams kp)
{
    extern __shared__ __align__(16) unsigned char smem[];
    fused_loop<BITS, NC, MSD>(kp, smem);
}
