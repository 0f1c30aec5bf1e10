// kmcg_fused.hip -- the fused step loop (one layer of local_smart processes,
// or lat_int with every group tabulated; one or two dimensions).
//
// Included by kmcg_engine.hip (device part, inside its namespace).
//
// A process that runs has every one of its conditions fulfilled (its lists
// match the lattice), so the species of all its condition sites are known
// before any lattice read, before and after each of its writes.  The
// library therefore folds the routines of one process into ONE flat list of
// updates, one lane's work each (build_fused, build_fused_li in
// kmcg_engine.hip):
//   local_smart: an update adds or deletes one (process, site) pair when its
//     conditions hold.  Updates that contradict the known species are gone,
//     conditions the known species fulfil are dropped; what is left reads
//     only sites the process does not write (ZGB keeps 15 updates per
//     process with at most one condition each, generic 17 with two; RuO2 38
//     with one, 45 with two).
//   lat_int: an update is one (group, cell) pair of the modified list; it
//     deletes the variant the group's table gives before the writes and adds
//     the one it gives after them.  Both lookups differ in a base only, the
//     open sites (at most four) are read once.
// The updates of one process (lat_int: of one group) are neighbouring
// lanes, in the reference's order, so the lane that owns a process finds its
// entries as a run of bits and fetches them with ds_bpermute: no mailboxes,
// no rounds of LDS atomics.
//
// What bounds a step is its chain of dependent instructions and latencies (a
// lone wave issues about one instruction in eight cycles): the read of the
// picked site, the evaluation, the list reads, the selection of the next
// process.  Deletions are of registered entries only (their conditions
// hold), so the counts after the step are known from the bits alone; the
// next step is selected from them and ITS site read issued before the list
// updates of this step run.  A slot the updates overwrite is patched in a
// register.
//
// Measured against the generic loops, per 1000 steps: ZGB 4096 x 128x128
// 5.41 -> 2.73 ms, RuO2 mix of 2048 5.42 -> 3.06 ms, RuO2 lat_int, 300 odd
// lattices 5.91 -> 2.25 ms, pairwise lat_int 512 x 256x256 4.48 -> 2.5 ms
// (kernel); one RuO2 64x64 trajectory 3.8 -> 1.56 us per step; tracking on
// the pairwise model (264 updates in five chunks) 14.1 -> 7.6 us per step.
//
// Record of one lane (RW words, 64 lanes per chunk, the chunks of a process
// in turn):
//   word 0: bits 0-6 row (P + process - 1), 7-12 first lane of the updates
//           of process (lane + 1), lat_int: of its group; 13-17 their number
//           (lat_int 13-16: this lane's place in its run), 18-21 condition
//           code, 22-25 and 26-29 species the lane's write takes away and
//           puts down (equal: no write), 31 the update deletes
//   FZ_1 (one condition):  site, condition site, write site
//   FZ_4 (four, chunks):   four condition codes | chunks << 16, site, four
//                          condition sites, write site
//   FZ_LI (lat_int):       cell, byte offsets of the two lookups (before |
//                          after << 16), four open sites, write site
// site word: (dx * spuck + n - n_exec) | dy << 16, signed halves, from the
// picked site; open site: the same in 12 and 7 bits | stride << 19.
// condition code: species + 1 for the 2-bit lattice, the species otherwise;
// a lane without an open condition tests a site the process knows, a lane
// without an update has code 15, which no site holds.

enum : int { FZ_1 = 1, FZ_LI = 2, FZ_4 = 4 };

template <int FORM>
struct FzRec {
    static constexpr int RW = FORM == FZ_1 ? 4 : 8;
    int w[RW];
    __device__ __forceinline__ int write_site() const { return w[RW - 1]; }
    __device__ __forceinline__ int site() const { return FORM == FZ_4 ? w[2] : w[1]; }
};

__device__ __forceinline__ int bf_s(int v, int off, int w) { return __builtin_amdgcn_sbfe(v, off, w); }
__device__ __forceinline__ int bf_u(int v, int off, int w) { return (int)__builtin_amdgcn_ubfe((unsigned)v, off, w); }

template <int FORM>
__device__ __forceinline__ void fz_load(const int *recs, int chunk, int lane, FzRec<FORM> &q)
{
    constexpr int RW = FzRec<FORM>::RW;
    const int4 *p = (const int4 *)(recs + (size_t)chunk * (64 * RW)) + lane * (RW / 4);
#pragma unroll
    for (int i = 0; i < RW / 4; ++i) {
        const int4 a = p[i];
        q.w[4 * i] = a.x;
        q.w[4 * i + 1] = a.y;
        q.w[4 * i + 2] = a.z;
        q.w[4 * i + 3] = a.w;
    }
}

// The picked site (uniform): its number, its place in its row of sX sites,
// its row.
struct FzAt {
    int s0, rem, y, sX, Y;
};

// the 0-based site at (lo, dy) from the picked one; IN: nothing wraps there
template <bool IN>
__device__ __forceinline__ int fz_site(const FzAt &p, int lo, int dy)
{
    if (IN)
        return __mul24(dy, p.sX) + (p.s0 + lo);
    return __mul24(wrap1(p.y + dy, p.Y), p.sX) + wrap1(p.rem + lo, p.sX);
}
template <bool IN>
__device__ __forceinline__ int fz_site(const FzAt &p, int w)
{
    return fz_site<IN>(p, (int)(short)(w & 0xFFFF), w >> 16);
}

// a site's species code as the records hold it
template <int BITS>
__device__ __forceinline__ int fz_code(const unsigned char *lat, int s)
{
    if (BITS == 8)
        return (int)lat[s];
    const unsigned w = ((const unsigned *)lat)[(unsigned)s >> 4];
    return (int)__builtin_amdgcn_ubfe(w, (unsigned)s << 1, 2);
}

// Does this lane's update take place (FZ_1, FZ_4)?  s: its site.
template <int BITS, int FORM, bool IN>
__device__ __forceinline__ bool fz_eval(const unsigned char *lat, const FzAt &p, const FzRec<FORM> &q, int &s, int &ws)
{
    constexpr int NC = FORM == FZ_1 ? 1 : 4, C0 = FORM == FZ_1 ? 2 : 3;
    int got[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c)
        got[c] = fz_code<BITS>(lat, fz_site<IN>(p, q.w[C0 + c]));
    s = fz_site<IN>(p, q.site());
    ws = fz_site<IN>(p, q.write_site());
    if (FORM == FZ_1)
        return got[0] == bf_u(q.w[0], 18, 4);
    int all = got[0];
#pragma unroll
    for (int c = 1; c < NC; ++c)
        all |= got[c] << (4 * c);
    return all == (q.w[1] & 0xFFFF);
}

// The variants this lane's (group, cell) pair has before and after the
// writes (FZ_LI; 0: none).
template <int BITS, bool IN>
__device__ __forceinline__ void fz_eval_li(const unsigned char *lat, const unsigned char *tab, const FzAt &p,
                                           const FzRec<FZ_LI> &q, int &s, int &ws, int &pd, int &pa)
{
    int got[4];
#pragma unroll
    for (int c = 0; c < 4; ++c)
        got[c] = fz_code<BITS>(lat, fz_site<IN>(p, bf_s(q.w[3 + c], 0, 12), bf_s(q.w[3 + c], 12, 7)));
    s = fz_site<IN>(p, q.site());
    ws = fz_site<IN>(p, q.write_site());
    int idx = 0;
#pragma unroll
    for (int c = 0; c < 4; ++c)
        idx = (int)__umul24(got[c], (unsigned)q.w[3 + c] >> 19) + idx;
    pd = tab[(q.w[2] & 0xFFFF) + idx];
    pa = tab[(int)((unsigned)q.w[2] >> 16) + idx];
}

// What one owner lane replays its updates with.
struct FzList {
    Rows L;
    int V;
    int pk;          // the slot the next step's site is read from (-1: another lane's list)
    int patch;       // its new content when an update of this step writes it
    int err;
};

// Up to RB updates of this lane's list, in order (add_proc/del_proc,
// base.mpy:211-301).  bits: this lane's entries, relative to lane a (LI: 16
// deletions, then 16 additions); ent: the update lanes' sites (+ bit 31: it
// deletes), bv0 their back-indices; t<j>: list slot nr - j.  Everything an
// entry may need from an earlier one of the block (the slot it wrote and
// the site it put there) stays in registers, so no entry waits for memory
// or LDS; every change is written through in order.  Each entry is two
// stores, and two more when the last site moves into a freed slot.  Every
// lane takes part.
template <int RB, bool LI>
__device__ __forceinline__ void fz_replay(FzList &F, int &nr, unsigned &bits, int a, int ent, int bv0, int t0, int t1,
                                          int t2, int t3)
{
    int st[RB], bv[RB];
    bool act[RB], isd[RB];
#pragma unroll
    for (int i = 0; i < RB; ++i) {
        act[i] = bits != 0;
        const int rel = __builtin_ctz(bits | 0x80000000u);
        const int src = (a + (LI ? rel & 15 : rel)) << 2;
        st[i] = __builtin_amdgcn_ds_bpermute(src, ent);
        bv[i] = __builtin_amdgcn_ds_bpermute(src, bv0);
        isd[i] = LI ? rel < 16 : st[i] < 0;
        if (!LI)
            st[i] &= 0x7FFFFFFF;
        bits &= bits - 1;
    }
    const int nr0 = nr;
    int cur = nr0;
    int ws[RB], wv[RB];
#pragma unroll
    for (int i = 0; i < RB; ++i) {
        // the last slot's site and the deleted site's place, as the entries
        // before left them
        int moved = t0;
        if (i > 0)
            moved = nr0 - cur == 1 ? t1 : moved;
        if (i > 1)
            moved = nr0 - cur == 2 ? t2 : moved;
        if (i > 2)
            moved = nr0 - cur == 3 ? t3 : moved;
#pragma unroll
        for (int j = 0; j < i; ++j)
            moved = ws[j] == cur ? wv[j] : moved;
        int mp = bv[i];
#pragma unroll
        for (int j = 0; j < i; ++j)
            mp = wv[j] == st[i] ? ws[j] : mp;
        // (lists that match the lattice never fail here)
        const bool okd = (unsigned)(mp - 1) < (unsigned)cur;
        const bool del = act[i] && isd[i] && okd;
        const bool add = act[i] && !isd[i] && cur < F.V;
        F.err |= act[i] && !del && !add ? 1 : 0;
        const bool mv = del && mp < cur;
        const int slot = del ? mp : cur + 1;
        const int val = del ? (mv ? moved : 0) : st[i];
        if (del || add) {
            F.L.b(st[i]) = del ? 0 : slot;
            F.L.s(slot) = val;
        }
        if (mv) {
            F.L.b(moved) = mp;
            F.L.s(cur) = 0;
        }
        const bool put = add || mv;
        ws[i] = put ? slot : 0;
        wv[i] = put ? val : 0;
        F.patch = ws[i] == F.pk ? wv[i] : F.patch;
        cur = del ? cur - 1 : add ? cur + 1 : cur;
    }
    nr = cur;
}

// The left-to-right FP64 prefix over lanes (accumulate) for a long chain.
// Lane l of L links from lane f on adds, at time t, the term of lane
// l - (L - 1) + t, read from LDS at consecutive addresses; terms below lane f
// read as zero (adding zero changes no bit), so every lane ends with its own
// term after the last link.  One LDS read serves two links and a link is one
// dependent addition, where the shifted form spends two shifts, a hazard
// and the addition.  `tz`: 128 doubles, the first 64 zero.
__device__ __forceinline__ double fz_chain(double *tz, double c, double acc, int P, int lane, int f)
{
    constexpr int U = 8;
    const int L = (P - f + U - 1) & ~(U - 1);
    const double before = f > 0 ? readlane_d(acc, f - 1) : 0.0;
    tz[64 + lane] = lane >= f ? c : 0.0;
    wave_sync();
    const double *p = tz + (64 + lane - (L - 1));
    double a = lane >= f ? before : acc;
    double v[U];
#pragma unroll
    for (int k = 0; k < U; ++k)
        v[k] = p[k];
    for (int k0 = U; k0 < L; k0 += U) {
        double vn[U];
#pragma unroll
        for (int k = 0; k < U; ++k)
            vn[k] = p[k0 + k];
#pragma unroll
        for (int k = 0; k < U; ++k)
            a = a + v[k];
#pragma unroll
        for (int k = 0; k < U; ++k)
            v[k] = vn[k];
    }
#pragma unroll
    for (int k = 0; k < U; ++k)
        a = a + v[k];
    wave_sync();
    return a;
}

// The kernel's parameters read again where they are needed, for the parts
// of the loop that seldom run: kept in scalar registers over the loop they
// would be spilled to vector lanes and back on every step.
typedef const __attribute__((address_space(4))) KParams *FzCold;
__device__ __forceinline__ FzCold fz_cold()
{
    FzCold p = (FzCold)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return p;
}

// One step's uniforms (-log(u_time), u_proc, u_site), called once in 64
// steps: a call, so that its constants take no registers in the loop.
struct FzUni {
    double mlog, u1, u2;
};
__device__ __attribute__((noinline)) FzUni fz_uniforms(unsigned seed, unsigned stream, unsigned long long step)
{
    double uu[3];
    step_uniforms(seed, stream, step, uu);
    return {-log(uu[0]), uu[1], uu[2]};
}

// do_kmc_steps for one replica per wave (proclist_generic_subroutines.mpy:
// 1-44).  The launch guarantees: records for the model, at most 64
// processes and two dimensions, lists matching the lattices, lattices in
// LDS, no extent below 2 * fz_moff + 1 (no two offsets of the records meet).
template <int BITS, int FORM, bool MSD>
__device__ __forceinline__ void fused_loop(const KParams &kp, unsigned char *smem)
{
    constexpr bool LI = FORM == FZ_LI;
    // lat_int: the groups' tables, one copy per workgroup
    if (LI) {
        const int *src = kp.fz_recs + kp.fz_tab_off;
        for (int i = threadIdx.x; i < kp.prog_lds / 4; i += blockDim.x)
            ((int *)smem)[i] = src[i];
        __syncthreads();
    }
    Wave<1, BITS> W;
    const int r = wave_setup<1, BITS, true, false>(W, kp, smem);
    if (r < 0)
        return;
    const int slot = blockIdx.x * kp.wpg + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = W.lane, P = W.P;
    const int *recs = kp.fz_recs;
    const int nch = FORM == FZ_4 ? kp.fz_nch : 1;
    double *tz = (double *)W.win;
    unsigned *bm = (unsigned *)(tz + 128);             // FZ_LI: entries per process
    tz[lane] = 0.0;
    if (LI)
        bm[lane] = 0;
    wave_sync();
    const int st0 = kp.status[r];
    long long n = kp.nsteps;
    if (kp.budget)
        n = min(n, kp.budget[slot]);
    if (st0 != ST_OK)
        n = 0;
    if (kp.srec)
        count_species<1, BITS>(W);
    double t = kp.ktime[r], dt_last = kp.kdt[r];
    int st = st0;
    long long done = 0, drawn = 0;                     // steps done, uniforms used
    int rec_left = kp.sample_every, rec_idx = 0;
    const unsigned row = (unsigned)W.V1 << 2;          // bytes of one list
    FzList F;
    F.L.base = (char *)W.avail;
    F.L.so = row * (unsigned)(lane < P ? lane : 0);
    F.L.bo = row * (unsigned)(P + (lane < P ? lane : 0));
    F.V = W.d.V;
    F.pk = -1;
    F.patch = 0;
    F.err = 0;
    FzAt at;
    at.sX = W.d.sX;
    at.Y = W.d.Y;
    const Magic mrow = make_magic(at.sX);
    const unsigned in_lo = W.d.moff * W.d.spuck, in_w = at.sX - 2 * in_lo;
    const unsigned in_y = W.d.dim >= 2 ? W.d.moff : 0, in_h = at.Y - 2 * in_y;
    double lmlog = 0.0, lu1 = 0.0, lu2 = 0.0;
    // the selected step: its terms, total, process, slot, site on the way
    double acc = 0.0, c = 0.0, total = 0.0, mlog = 0.0;
    int pick = 0, kk = 0, sv = 0;
    int nr = W.nr[0], nrs = nr;                        // nrs: the counts acc belongs to
    const double rate = W.rate[0];
    double integ = W.integ[0];
    FzRec<FORM> q;
    // selects step k (0-based in this run) after the counts nrx: accum_rates,
    // process, slot; its site and records are requested, not waited for
    auto select = [&](long long k, int nrx, bool anew) {
        const int uj = (int)k & 63;
        if (uj == 0) {
            // uniforms of 64 steps at a time: lane i draws step k + i
            const FzCold kc = fz_cold();
            const FzUni u = fz_uniforms(kc->seed[r], kc->stream[r], kc->rngctr[r] + (unsigned long long)k + lane);
            lmlog = u.mlog;
            lu1 = u.u1;
            lu2 = u.u2;
        }
        c = (double)nrx * rate;
        const unsigned long long ch = __ballot(nrx != nrs);
        nrs = nrx;
        int f = ch ? __ffsll((long long)ch) - 1 : 64;
        if (anew)
            f = 0;
        if (P - f > 6) {
            acc = fz_chain(tz, c, acc, P, lane, f);
        } else if (f < P) {
            const double cs[1] = {c};
            double as[1] = {acc};
            const int fs[1] = {f};
            accumulate<1>(cs, as, P, lane, fs);
            acc = as[0];
        }
        total = readlane_d(acc, P - 1);
        mlog = readlane_d(lmlog, uj);
        if (total > 0.0) {
            // interval_search_real (base.mpy:1234-1338): the first process
            // whose prefix exceeds the value (no equal prefix lies left of
            // it), past the end the leftmost of those equal to the last
            const double value = readlane_d(lu1, uj) * total;
            unsigned long long mk = __ballot(lane < P && value < acc);
            if (!mk)
                mk = __ballot(lane < P && acc == total);
            pick = __ffsll((long long)mk) - 1;
            const int nrp = readlane_i(nrx, pick);
            kk = (int)(1.0 + readlane_d(lu2, uj) * (double)nrp);
            kk = __builtin_amdgcn_readfirstlane(kk > nrp ? nrp : kk);
            F.pk = lane == pick && kk > 0 ? kk : -1;
            F.patch = 0;
            sv = *(const int *)(F.L.base + (row * (unsigned)pick + ((unsigned)max(kk, 0) << 2)));
            fz_load<FORM>(recs, pick * nch, lane, q);
        }
    };
    if (n > 0) {
        select(0, nr, true);
        drawn = 0;
    }
#if KMCG_PHASES
    for (int i = 0; i < 5; ++i)
        W.tph[i] = 0;
    W.nblk = W.napply = 0;
    W.tmark = __builtin_amdgcn_s_memtime();
#endif
    while (done != n) {
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
        const double ctotal = total, cc = c, cmlog = mlog;
        drawn = done + 1;
        if (kk < 1) {                       // only a corrupted database gets here
            st = ST_CORRUPT;
            dt_last = cmlog / ctotal;
            t = t + dt_last;
            integ = integ + cc * dt_last;
            break;
        }
        at.s0 = site - 1;
        at.y = divm(at.s0, mrow);
        at.rem = at.s0 - at.y * at.sX;
        const bool inside = (unsigned)at.rem - in_lo < in_w && (unsigned)at.y - in_y < in_h;
        const int nchp = FORM == FZ_4 ? __builtin_amdgcn_readfirstlane(bf_u(q.w[1], 16, 5)) : 1;
        for (int ci = 0; ci < nchp; ++ci) {
            // evaluation; bits: this owner lane's entries, nd of them deletions
            int s, ws, a, nd, ent;
            unsigned bits, bo;
            bool back;
            if constexpr (LI) {
                int pd, pa;
                if (inside)
                    fz_eval_li<BITS, true>(W.lat.p, smem, at, q, s, ws, pd, pa);
                else
                    fz_eval_li<BITS, false>(W.lat.p, smem, at, q, s, ws, pd, pa);
                const unsigned at1 = 1u << bf_u(q.w[0], 13, 4);
                if (pd)
                    atomicOr(&bm[pd - 1], at1);
                if (pa)
                    atomicOr(&bm[pa - 1], at1 << 16);
                wave_sync();
                bits = bm[lane];
                wave_sync();
                bm[lane] = 0;
                a = bf_u(q.w[0], 7, 6);
                back = pd != 0;
                bo = (__umul24(P - 1 + pd, (unsigned)W.V1) + (unsigned)s + 1u) << 2;
                ent = s + 1;
                nd = __popc(bits & 0xFFFFu);
            } else {
                bool ok;
                if (inside)
                    ok = fz_eval<BITS, FORM, true>(W.lat.p, at, q, s, ws);
                else
                    ok = fz_eval<BITS, FORM, false>(W.lat.p, at, q, s, ws);
                back = ok && q.w[0] < 0;
                const unsigned long long mk = __ballot(ok), dk = __ballot(back);
                bo = (__umul24(q.w[0] & 127, (unsigned)W.V1) + (unsigned)s + 1u) << 2;
                a = bf_u(q.w[0], 7, 6);
                const int len = bf_u(q.w[0], 13, 5);
                bits = (unsigned)bf_u((int)(mk >> a), 0, len);
                nd = __popc((unsigned)bf_u((int)(dk >> a), 0, len));
                ent = (s + 1) | (q.w[0] & (int)0x80000000);
            }
            // back[site] of a deletion, the slots a deletion takes the last
            // site from
            int bv = 0;
            if (back)
                bv = *(const int *)(F.L.base + bo);
            const int ne = __popc(bits);
            const bool two = __ballot(ne > 1), three = __ballot(ne > 2), four = __ballot(ne > 3);
            int t0 = 0, t1 = 0, t2 = 0, t3 = 0;
            if (nd > 0)
                t0 = F.L.s(nr);
            if (two && nd > 1) {
                t1 = F.L.s(max(nr - 1, 0));
                if (nd > 2)
                    t2 = F.L.s(max(nr - 2, 0));
                if (nd > 3)
                    t3 = F.L.s(max(nr - 3, 0));
            }
            const int w0 = q.w[0];
            const bool lastc = ci == nchp - 1;
            PH_MARK(W, 2);
            if (lastc)
                select(done + 1, nr + ne - 2 * nd, false);
            else
                fz_load<FORM>(recs, cpick * nch + ci + 1, lane, q);
            PH_MARK(W, 0);
            // the writes (their old species are known); nothing of this
            // step reads a written site
            const int so = bf_u(w0, 22, 4), sn = bf_u(w0, 26, 4);
            if (so != sn) {
                W.lat.xset(ws, so, sn);
                if (W.track) {
                    const int tt = ws - divm(ws, W.ms) * W.d.spuck;
                    if (so < W.S)
                        atomicAdd(&W.occ[so * W.d.spuck + tt], -1);
                    if (sn < W.S)
                        atomicAdd(&W.occ[sn * W.d.spuck + tt], 1);
                }
            }
            wave_sync();
            if (lastc) {
                // update_clocks, update_integ_rate with the counts before
                const double dt = cmlog / ctotal;
                t = t + dt;
                dt_last = dt;
                integ = integ + cc * dt;
                W.pstat[0] += lane == cpick ? 1 : 0;
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
                fz_replay<4, LI>(F, nr, bits, a, ent, bv, t0, t1, t2, t3);
                while (__ballot(bits != 0)) {
#if KMCG_PHASES
                    W.nblk += 1;
#endif
                    // the next four: list tail and back-indices read again,
                    // behind the stores of the block before
                    const bool more = bits != 0;
                    t0 = more ? F.L.s(nr) : 0;
                    t1 = more ? F.L.s(max(nr - 1, 0)) : 0;
                    t2 = more ? F.L.s(max(nr - 2, 0)) : 0;
                    t3 = more ? F.L.s(max(nr - 3, 0)) : 0;
                    if (back)
                        bv = *(const int *)(F.L.base + bo);
                    fz_replay<4, LI>(F, nr, bits, a, ent, bv, t0, t1, t2, t3);
                }
            } else if (three) {
                fz_replay<3, LI>(F, nr, bits, a, ent, bv, t0, t1, t2, 0);
            } else if (two) {
                fz_replay<2, LI>(F, nr, bits, a, ent, bv, t0, t1, 0, 0);
            } else {
                fz_replay<1, LI>(F, nr, bits, a, ent, bv, t0, 0, 0, 0);
            }
            PH_MARK(W, 3);
        }
        if (MSD && kp.acf_pa && lane == 0)
            acf_after(kp, r);
        if (__ballot(F.err)) {
            st = LI ? ST_DEL_ABSENT : ST_CORRUPT;
            break;
        }
        if (W.track && --rec_left == 0) {
            const FzCold kc = fz_cold();
            W.integ[0] = integ;
            write_record<1, BITS>(W, kp, slot, rec_idx, t, dt_last, kc->kstep[r] + done, ST_OK);
            rec_left = kc->sample_every;
            rec_idx += 1;
        }
    }
    W.nr[0] = nr;
    W.integ[0] = integ;
    const FzCold kc = fz_cold();
    steps_end<1, BITS, true>(W, kp, r, slot, t, dt_last, kc->kstep[r] + drawn, kc->rngctr[r] + drawn, st, done);
}

template <int BITS, int FORM, bool MSD>
__global__ __launch_bounds__(64 * MAX_WPG) __attribute__((amdgpu_waves_per_eu(4))) void kmc_steps_kernel_fz(KParams kp)
{
    extern __shared__ __align__(16) unsigned char smem[];
    fused_loop<BITS, FORM, MSD>(kp, smem);
}
