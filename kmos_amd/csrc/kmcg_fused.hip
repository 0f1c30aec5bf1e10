// kmcg_fused.hip -- the fused step loop (local_smart processes on one or
// several layers, or one layer of lat_int with every group tabulated; one or
// two dimensions).
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
// 5.42 -> 2.22 ms, RuO2 mix of 2048 5.42 -> 2.60 ms, RuO2 lat_int, 300 odd
// lattices 5.95 -> 1.79 ms, pairwise lat_int 512 x 256x256 4.48 -> 1.85 ms
// (kernel, the first steps after an empty lattice), Pd oxide on two layers
// (25 sites per cell) 4.54 -> 1.62 ms; one RuO2 64x64 trajectory 3.8 -> 1.24
// us per step; the pairwise model as local_smart (264 updates in five
// chunks) with moves tracked 14.1 -> 4.5 us per step.
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
//   FZ_M (several layers): as FZ_4.  The lists of several local_smart layers
//                          promise only that registered processes hold: a
//                          deletion that finds no entry is none (the next
//                          step is then selected again), and a write whose
//                          old species no condition names (word 0, bit 30)
//                          looks before the step; where it fails the run
//                          stops short and the generic loop behind it
//                          finishes it.
//   FZ_LI (lat_int):       cell, byte offsets of the two lookups (before |
//                          after << 16), four open sites, write site
// site word: (dx * spuck + n - n_exec) | dy << 16, signed halves, from the
// picked site; open site: the same in 12 and 7 bits | stride << 19.
// condition code: species + 1 for the 2-bit lattice, the species otherwise;
// a lane without an open condition tests a site the process knows, a lane
// without an update has code 15, which no site holds.

enum : int { FZ_1 = 1, FZ_LI = 2, FZ_M = 3, FZ_4 = 4 };
__host__ __device__ constexpr bool fz_wide(int form) { return form == FZ_4 || form == FZ_M; }

template <int FORM>
struct FzRec {
    static constexpr int RW = FORM == FZ_1 ? 4 : 8;
    int w[RW];
    __device__ __forceinline__ int write_site() const { return w[RW - 1]; }
    __device__ __forceinline__ int site() const { return fz_wide(FORM) ? w[2] : w[1]; }
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

// species old -> v at site s by exclusive or, lanes with old == v on a spare
// word of their own (no divergent region); other lanes may write other
// sites of the same word
template <int BITS>
__device__ __forceinline__ void fz_write(unsigned char *lat, unsigned *spare, int s, int old, int v)
{
    unsigned *w = (unsigned *)lat + ((unsigned)s >> (BITS == 8 ? 2 : 4));
    const unsigned x = BITS == 8 ? (unsigned)(old ^ v) << ((s & 3) * 8)
                                 : (unsigned)((old + 1) ^ (v + 1)) << ((s << 1) & 31);
    atomicXor(old != v ? w : spare, x);
}

// What a lane's record names around the picked site: its update's site, the
// site it writes, the sites it tests.  The plain form first, without a
// branch; near the faces the sites are formed again, wrapped.
template <int FORM>
struct FzSites {
    static constexpr int NC = FORM == FZ_1 ? 1 : 4;
    int s, ws, cs[NC];
    template <bool IN>
    __device__ __forceinline__ void form(const FzAt &p, const FzRec<FORM> &q)
    {
        s = fz_site<IN>(p, q.site());
        ws = fz_site<IN>(p, q.write_site());
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            const int w = q.w[FORM == FZ_1 ? 2 : 3 + c];
            cs[c] = FORM == FZ_LI ? fz_site<IN>(p, bf_s(w, 0, 12), bf_s(w, 12, 7)) : fz_site<IN>(p, w);
        }
    }
    // Does this lane's update take place (FZ_1, FZ_4)?
    template <int BITS>
    __device__ __forceinline__ bool holds(const unsigned char *lat, const FzRec<FORM> &q) const
    {
        int all = fz_code<BITS>(lat, cs[0]);
#pragma unroll
        for (int c = 1; c < NC; ++c)
            all |= fz_code<BITS>(lat, cs[c]) << (4 * c);
        return all == (FORM == FZ_1 ? bf_u(q.w[0], 18, 4) : (q.w[1] & 0xFFFF));
    }
    // The variants this lane's (group, cell) pair has before and after the
    // writes (FZ_LI; 0: none).
    template <int BITS>
    __device__ __forceinline__ void variants(const unsigned char *lat, const unsigned char *tab,
                                             const FzRec<FORM> &q, int &pd, int &pa) const
    {
        int got[NC], idx = 0;
#pragma unroll
        for (int c = 0; c < NC; ++c)
            got[c] = fz_code<BITS>(lat, cs[c]);
#pragma unroll
        for (int c = 0; c < NC; ++c)
            idx = (int)__umul24(got[c], (unsigned)q.w[FORM == FZ_1 ? 0 : 3 + c] >> 19) + idx;
        pd = tab[(q.w[2] & 0xFFFF) + idx];
        pa = tab[(int)((unsigned)q.w[2] >> 16) + idx];
    }
};

// A replica's lists through a buffer descriptor: a lane whose offset is
// FZ_NONE lies outside it, so its load returns 0 and its store is dropped by
// the hardware's range check.  An access of some lanes costs one select that
// way (8 cycles of a lone wave) where a divergent region costs compare,
// save, branch and restore (45), and the code stays straight, so that the
// wait for the next step's site does not wait for the stores behind it.
constexpr unsigned FZ_NONE = 0x80000000u;
constexpr unsigned FZ_LEAD = 16;     // bytes before the first list (the pool's leading words or another list)
typedef int int4v __attribute__((ext_vector_type(4)));

// What one owner lane replays its updates with.
struct FzList {
    unsigned so, bo; // byte offsets of this lane's sites[p] and back[p]
    int V;
    int pk;          // the slot the next step's site is read from (-1: another lane's list)
    int patch;       // its new content when an update of this step writes it
    int err;
};

// Entries [I0, I0 + N) of a block of this lane's updates, in order
// (add_proc/del_proc, base.mpy:211-301).  bits: this lane's entries,
// relative to lane a (LI: 16 deletions, then 16 additions); ent: the update
// lanes' sites (+ bit 31: it deletes), bv0 their back-indices; t<j>: list
// slot nr0 - j.  Everything an entry may need from an earlier one of the
// block (the slot it wrote and the site it put there) stays in registers,
// so no entry waits for memory; every change is written through in order.
// A lane without an entry changes nothing.  Every lane takes part.
struct FzBlock {
    int nr0, ws[4], wv[4];
};
template <int I0, int N, int FORM>
__device__ __forceinline__ void fz_replay(__amdgpu_buffer_rsrc_t rs, FzList &F, FzBlock &B, int &nr, unsigned &bits,
                                          int a, int ent, int bv0, int t0, int t1, int t2, int t3)
{
    constexpr bool LI = FORM == FZ_LI;
    int st[N], bv[N];
    bool act[N], isd[N];
#pragma unroll
    for (int i = 0; i < N; ++i) {
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
    int cur = nr;
#pragma unroll
    for (int i = 0; i < N; ++i) {
        // the last slot's site and the deleted site's place, as the entries
        // before left them
        int moved = t0;
        if (I0 + i > 0)
            moved = B.nr0 - cur == 1 ? t1 : moved;
        if (I0 + i > 1)
            moved = B.nr0 - cur == 2 ? t2 : moved;
        if (I0 + i > 2)
            moved = B.nr0 - cur == 3 ? t3 : moved;
        int mp = bv[i];
#pragma unroll
        for (int j = 0; j < I0 + i; ++j) {
            moved = B.ws[j] == cur ? B.wv[j] : moved;
            mp = B.wv[j] == st[i] ? B.ws[j] : mp;
        }
        // (lists that match the lattice never fail here)
        const bool okd = (unsigned)(mp - 1) < (unsigned)cur;
        const bool del = act[i] && isd[i] && okd;
        const bool add = act[i] && !isd[i] && cur < F.V;
        F.err |= act[i] && !del && !add && !(FORM == FZ_M && isd[i] && mp == 0) ? 1 : 0;
        const bool mv = del && mp < cur, put = add || mv;
        const int slot = del ? mp : cur + 1;
        const int val = del ? moved : st[i];
        // back[site], the slot, back[moved site]; slots past the end keep
        // what they held
        __builtin_amdgcn_raw_buffer_store_b32(del ? 0 : slot, rs,
                                              del || add ? F.bo + ((unsigned)st[i] << 2) : FZ_NONE, 0, 0);
        __builtin_amdgcn_raw_buffer_store_b32(val, rs, put ? F.so + ((unsigned)slot << 2) : FZ_NONE, 0, 0);
        __builtin_amdgcn_raw_buffer_store_b32(slot, rs, mv ? F.bo + ((unsigned)moved << 2) : FZ_NONE, 0, 0);
        B.ws[I0 + i] = put ? slot : 0;
        B.wv[I0 + i] = put ? val : 0;
        F.patch = put && slot == F.pk ? val : F.patch;
        cur = del ? cur - 1 : add ? cur + 1 : cur;
    }
    nr = cur;
}

// The left-to-right FP64 prefix over lanes (accumulate).  Lane l of L links
// from lane f on adds, at time t, the term of lane l - (L - 1) + t, read from
// LDS at consecutive addresses; terms below lane f read as zero (adding zero
// changes no bit), so every lane ends with its own term after the last link.
// One LDS read serves two links and a link is one dependent addition (9
// cycles), where the shifted form spends two shifts, their hazard and the
// addition (about 40).  `tz`: 128 doubles, the first 64 zero.
__device__ __forceinline__ double fz_chain(double *tz, double c, double acc, int P, int lane, int f)
{
    constexpr int U = 8;
    const int L = max(P - f + U - 1, U) & ~(U - 1);
    const double before = readlane_d(acc, max(f, 1) - 1);
    tz[64 + lane] = lane >= f ? c : 0.0;
    wave_sync();
    const double *p = tz + (64 + lane - (L - 1));
    double a = lane >= f ? (f > 0 ? before : 0.0) : acc;
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

// What a run keeps beside the steps.
enum : int { FZ_PLAIN = 0, FZ_REC = 1, FZ_MSD = 2 };

// The particle moves of a displacement run (msd_track has the steps in
// order).  msd_track waits for the hop's table entry, the particle at the
// hop's start, its displacement and the event counter one after the other,
// four trips to memory that a lone wave has nothing to hide behind.  Here
// the hop is requested with the step's records and the particle as soon as
// the site is known; what needs its number is written one step later, after
// the list updates, whose loads are younger than it.  The displacement is a
// memory atomic (one add, rounded as the add of a register), so nothing waits
// for it; the events are counted in a register.  Measured (pairwise
// local_smart 128x128 x32, 4000 steps): 4.5 us per step where a plain run
// takes 3.9; with msd_track in its place 5.6.
struct FzMove
{
    int h0, dx, dy, dz, n;           // the hop of the process, lane 0: from, else to
    double d;                        // lane 0..2: its displacement
    int p, fin;                      // the step before: its particle, the site it went to
    bool hop, open;                  // ... whether it was a hop; whether there is one to write
    long long ev, ev_n;              // events so far, and room for them
};

__device__ __forceinline__ void fz_move_load(const KParams &kp, int pick, int lane, FzMove &m)
{
    const int *h = kp.msd_hop + MSD_HOP_W * pick;
    m.h0 = h[0];
    const int *e = h + (lane == 0 ? 1 : 5);
    m.dx = e[0];
    m.dy = e[1];
    m.dz = e[2];
    m.n = e[3];
    m.d = kp.msd_d[3 * pick + min(lane, 2)];
}

// the step at `site`: its particle requested, its place emptied
template <int BITS>
__device__ __forceinline__ void fz_move_open(const Wave<1, BITS> &W, const KParams &kp, long long o, int site, FzMove &m)
{
    m.open = true;
    m.hop = __builtin_amdgcn_readfirstlane(m.h0) != 0;
    m.p = m.fin = 0;
    if (!m.hop)
        return;
    const int s0 = site - 1;
    const int cell = divm(s0, W.ms);
    const int yz = divm(cell, W.mx);
    const int z = divm(yz, W.my);
    const int at = site0(W.d, cell - yz * W.d.X, yz - z * W.d.Y, z, m.dx, m.dy, m.dz, m.n) + 1;
    const int init = readlane_i(at, 0);
    m.fin = readlane_i(at, 1);
    int *id = kp.msd_id + o;
    m.p = id[init];
    if (W.lane == 0)
        id[init] = 0;
}

__device__ __forceinline__ void fz_move_close(const KParams &kp, int r, long long o, int lane, double d, FzMove &m)
{
    if (!m.open)
        return;
    m.open = false;
    if (m.hop) {
        if (lane < 3)
            unsafeAtomicAdd(kp.msd_disp + 3 * (o + m.p) + lane, d);
        if (lane == 0) {
            kp.msd_id[o + m.fin] = m.p;
            int *sa = kp.msd_site + o;
            sa[m.p] = m.fin;
            sa[0] = 0;
        }
    }
    if (m.ev < m.ev_n) {
        int *ev = kp.msd_ev + 2 * ((long long)r * m.ev_n + m.ev);
        if (lane == 0) {
            ev[0] = m.p;
            ev[1] = m.fin;
        }
        m.ev += 1;
    }
}

// do_kmc_steps for one replica per wave (proclist_generic_subroutines.mpy:
// 1-44).  The launch guarantees: records for the model, at most 64
// processes and two dimensions, lists matching the lattices, lattices in
// LDS, no extent below 2 * fz_moff + 1 (no two offsets of the records meet),
// rows of more than one site, V times the row below 2^32.
//
// A lone wave issues an instruction in 6 to 9 cycles, and a branch or a
// divergent region costs 30 to 45: the loop has one pass per step with few
// branches, conditions end in selects, and stops (no process possible, a
// corrupted list) lower the limit the loop runs to.
template <int BITS, int FORM, int MODE>
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
    const int rslot = blockIdx.x * kp.wpg + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = W.lane, P = W.P;
    const int *recs = kp.fz_recs;
    const int nch = fz_wide(FORM) ? kp.fz_nch : 1;
    double *tz = (double *)W.win;
    unsigned *bm = (unsigned *)(tz + 128);             // FZ_LI: entries per process, then spare words
    tz[lane] = 0.0;
    if (LI)
        bm[lane] = 0;
    wave_sync();
    int st = kp.status[r];
    long long n = kp.nsteps;
    if (kp.budget)
        n = min(n, kp.budget[rslot]);
    if (st != ST_OK)
        n = 0;
    if (MODE == FZ_REC)
        count_species<1, BITS>(W);
    double t = kp.ktime[r];
    int rec_left = kp.sample_every + 1, rec_idx = 0;
    const unsigned row = (unsigned)W.V1 << 2;          // bytes of one list
    FzList F;
    const __amdgpu_buffer_rsrc_t rs =
        __builtin_amdgcn_make_buffer_rsrc((char *)W.avail - FZ_LEAD, 0, (int)(2u * P * row + FZ_LEAD), 0x00027000);
    F.so = FZ_LEAD + row * (unsigned)(lane < P ? lane : 0);
    F.bo = FZ_LEAD + row * (unsigned)(P + (lane < P ? lane : 0));
    F.V = W.d.V;
    F.pk = -1;
    F.patch = 0;
    F.err = 0;
    FzAt at;
    at.sX = W.d.sX;
    at.Y = W.d.Y;
    const unsigned mrow = make_magic(at.sX).m;         // (the launch: 1 < sX, V * sX < 2^32)
    const unsigned in_lo = __builtin_amdgcn_readfirstlane(W.d.moff * W.d.spuck);
    const unsigned in_y = __builtin_amdgcn_readfirstlane(W.d.dim >= 2 ? W.d.moff : 0);
    const unsigned in_w = __builtin_amdgcn_readfirstlane(at.sX - 2 * in_lo);
    const unsigned in_h = __builtin_amdgcn_readfirstlane(at.Y - 2 * in_y);
    const double rate = W.rate[0];
    double integ = W.integ[0];
    int nr = W.nr[0];
    double lmlog = 0.0, lu1 = 0.0, lu2 = 0.0;
    double acc = 0.0;
    int nrs = -1;                    // the counts acc belongs to (none yet)
    int nrx = nr;                    // the counts after the step before
    // the step before: its entries in this lane's list, its terms (none yet)
    unsigned bits = 0, bo = 0;
    int a = 0, ent = 0, bv = 0, t0 = 0, t1 = 0, t2 = 0, t3 = 0;
    bool back = false, three = false;
    double cc = 0.0, cmlog = 0.0, ctotal = 1.0;
    int cpick = -1;
    double total = 0.0;
    int kk = 0;
    bool bail = false;               // FZ_M: step k is left to the generic loop
    double dt_done = 0.0;            // FZ_M: the last finished step's duration
    FzRec<FORM> q;
    FzMove mv;
    double mv_d = 0.0;               // the displacement of the step before
    const bool moves = MODE == FZ_MSD && !kp.acf_pa;
    const long long mo = MODE == FZ_MSD ? kp.msd_off[r] : 0;
    mv.hop = mv.open = false;
    mv.h0 = mv.p = mv.fin = 0;
    mv.d = 0.0;
    mv.ev = mv.ev_n = 0;
    if (moves) {
        mv.ev_n = kp.msd_evcap;
        mv.ev = mv.ev_n > 0 ? kp.msd_evn[r] : 0;
    }
#if KMCG_PHASES
    for (int i = 0; i < 5; ++i)
        W.tph[i] = 0;
    W.nblk = W.napply = 0;
    W.tmark = __builtin_amdgcn_s_memtime();
#endif
    auto finish = [&]() {
        // the list updates of the step before
        FzBlock B;
        B.nr0 = nr;
        fz_replay<0, 2, FORM>(rs, F, B, nr, bits, a, ent, bv, t0, t1, t2, t3);
        if (three) {
            fz_replay<2, 2, FORM>(rs, F, B, nr, bits, a, ent, bv, t0, t1, t2, t3);
            while (__ballot(bits != 0)) {
#if KMCG_PHASES
                W.nblk += 1;
#endif
                // four more: the list tail and the back-indices read again,
                // behind the stores of the block before
                const int4v tl = __builtin_amdgcn_raw_buffer_load_b128(
                    rs, bits ? F.so + ((unsigned)nr << 2) - 12 : FZ_NONE, 0, 0);
                const int bn = __builtin_amdgcn_raw_buffer_load_b32(rs, back ? bo : FZ_NONE, 0, 0);
                B.nr0 = nr;
                fz_replay<0, 4, FORM>(rs, F, B, nr, bits, a, ent, bn, tl.w, tl.z, tl.y, tl.x);
            }
        }
#if KMCG_PHASES
        W.napply += 1;
        W.nblk += 1;
#endif
    };
    long long k = 0;                 // the step being selected
    long long limit = n;
    while (n > 0) {
        PH_MARK(W, 4);
        const int uj = (int)k & 63;
        if (uj == 0) {
            // uniforms of 64 steps at a time: lane i draws step k + i
            const FzCold kc = fz_cold();
            const FzUni u = fz_uniforms(kc->seed[r], kc->stream[r], kc->rngctr[r] + (unsigned long long)k + lane);
            lmlog = u.mlog;
            lu1 = u.u1;
            lu2 = u.u2;
        }
        // ---- select step k: accum_rates, process, slot; its site and
        // records are requested, not waited for
        const double c = (double)nrx * rate;
        const unsigned long long ch = __ballot(nrx != nrs);
        nrs = nrx;
        const int f = ch ? __ffsll((long long)ch) - 1 : 64;
        if (P > 2)
            acc = fz_chain(tz, c, acc, P, lane, f);
        else
            acc = wave_shr1z(c) + c;         // one link
        total = readlane_d(acc, P - 1);
        // interval_search_real (base.mpy:1234-1338): the first process whose
        // prefix exceeds the value (no equal prefix lies left of it), past
        // the end the leftmost of those equal to the last
        const double value = readlane_d(lu1, uj) * total;
        const unsigned long long mk = __ballot(lane < P && (value < acc || acc == total));
        const int pick = __ffsll((long long)mk) - 1;
        const int nrp = readlane_i(nrx, pick);
        kk = (int)(1.0 + readlane_d(lu2, uj) * (double)nrp);
        kk = __builtin_amdgcn_readfirstlane(kk > nrp ? nrp : kk);
        F.pk = lane == pick && kk > 0 ? kk : -1;
        F.patch = 0;
        const int sv = __builtin_amdgcn_raw_buffer_load_b32(
            rs, FZ_LEAD + row * (unsigned)pick + ((unsigned)max(kk, 0) << 2), 0, 0);
        fz_load<FORM>(recs, pick * nch, lane, q);
        if (moves)
            fz_move_load(kp, pick, lane, mv);
        limit = total > 0.0 && kk > 0 ? limit : k;
        PH_MARK(W, 0);
        // ---- finish step k - 1: update_clocks, update_integ_rate (with the
        // counts before it), its list updates
        if (MODE != FZ_MSD) {
            const double dt = cmlog / ctotal;
            if (FORM == FZ_M)
                dt_done = cpick >= 0 ? dt : dt_done;
            t = t + dt;
            integ = integ + cc * dt;
            W.pstat[0] += lane == cpick ? 1 : 0;
        }
        finish();
        if (moves)
            fz_move_close(kp, r, mo, lane, mv_d, mv);
        if (FORM == FZ_M && __ballot(nr != nrs)) {
            // a deletion found no entry: step k selected again from the
            // counts there are, nothing of step k - 1 left to do
            nrx = nr;
            bits = 0;
            back = three = false;
            cc = cmlog = 0.0;
            ctotal = 1.0;
            cpick = -1;
            limit = n;
            continue;
        }
        if (MODE == FZ_REC && --rec_left == 0) {
            const FzCold kc = fz_cold();
            W.integ[0] = integ;
            write_record<1, BITS>(W, kp, rslot, rec_idx, t, cmlog / ctotal, kc->kstep[r] + k, ST_OK);
            rec_left = kc->sample_every;
            rec_idx += 1;
        }
        PH_MARK(W, 3);
        if (k == limit || __ballot(F.err))
            break;
        // ---- step k: its site, read ahead or just written by the step before
        const int pv = readlane_i(F.patch, pick), sr = __builtin_amdgcn_readfirstlane(sv);
        const int site = pv ? pv : sr;
        PH_MARK(W, 1);
        cc = c;
        cmlog = readlane_d(lmlog, uj);
        ctotal = total;
        cpick = pick;
        at.s0 = site - 1;
        at.y = (int)__umulhi((unsigned)at.s0, mrow);
        at.rem = at.s0 - at.y * at.sX;
        const bool inside = (unsigned)at.rem - in_lo < in_w && (unsigned)at.y - in_y < in_h;
        if (MODE == FZ_MSD) {
            const double dt = cmlog / ctotal;
            t = t + dt;
            integ = integ + cc * dt;
            W.pstat[0] += lane == pick ? 1 : 0;
            if (kp.acf_pa)
                acf_before<1, BITS>(W, kp, r, t, dt, pick, site);
            else {
                mv_d = mv.d;
                fz_move_open<BITS>(W, kp, mo, site, mv);
            }
        }
        const int nchp = fz_wide(FORM) ? __builtin_amdgcn_readfirstlane(bf_u(q.w[1], 16, 5)) : 1;
        for (int ci = 0; ; ++ci) {
            // evaluation; bits: this owner lane's entries, nd of them deletions
            FzSites<FORM> z;
            z.template form<true>(at, q);
            if (!inside)
                z.template form<false>(at, q);
            int nd;
            if (FORM == FZ_M) {
                const int want = bf_u(q.w[0], 22, 4) + (BITS == 2 ? 1 : 0);
                if (__ballot(((q.w[0] >> 30) & 1) && fz_code<BITS>(W.lat.p, z.ws) != want)) {
                    bail = true;
                    break;
                }
            }
            a = bf_u(q.w[0], 7, 6);
            if constexpr (LI) {
                int pd, pa;
                z.template variants<BITS>(W.lat.p, smem, q, pd, pa);
                const unsigned at1 = 1u << bf_u(q.w[0], 13, 4);
                // (a lane without an entry has a spare word of its own)
                atomicOr(&bm[pd ? pd - 1 : 64 + lane], at1);
                atomicOr(&bm[pa ? pa - 1 : 64 + lane], at1 << 16);
                wave_sync();
                bits = bm[lane];
                wave_sync();
                bm[lane] = 0;
                back = pd != 0;
                bo = ((__umul24(P - 1 + pd, (unsigned)W.V1) + (unsigned)z.s) << 2) + (FZ_LEAD + 4);
                ent = z.s + 1;
                nd = __popc(bits & 0xFFFFu);
            } else {
                const bool ok = z.template holds<BITS>(W.lat.p, q);
                back = ok && q.w[0] < 0;
                const unsigned long long mo = __ballot(ok), mb = __ballot(back);
                bo = ((__umul24(q.w[0] & 127, (unsigned)W.V1) + (unsigned)z.s) << 2) + (FZ_LEAD + 4);
                const int len = bf_u(q.w[0], 13, 5);
                bits = (unsigned)bf_u((int)(mo >> a), 0, len);
                nd = __popc((unsigned)bf_u((int)(mb >> a), 0, len));
                ent = (z.s + 1) | (q.w[0] & (int)0x80000000);
            }
            // back[site] of a deletion; the slots a deletion takes the last
            // site from, read at once (the words before a list's first are
            // another list's or the pool's leading words)
            bv = __builtin_amdgcn_raw_buffer_load_b32(rs, back ? bo : FZ_NONE, 0, 0);
            const int4v tl = __builtin_amdgcn_raw_buffer_load_b128(
                rs, nd > 0 ? F.so + ((unsigned)nr << 2) - 12 : FZ_NONE, 0, 0);
            t0 = tl.w;
            t1 = tl.z;
            t2 = tl.y;
            t3 = tl.x;
            const int ne = __popc(bits);
            nrx = nr + ne - 2 * nd;
            three = __ballot(ne > 2) != 0;
            // the writes (their old species are known); nothing of this
            // step reads a written site
            const int so = bf_u(q.w[0], 22, 4), sn = bf_u(q.w[0], 26, 4);
            fz_write<BITS>(W.lat.p, bm + 64 + lane, z.ws, so, sn);
            if (MODE == FZ_REC && so != sn) {
                const int tt = z.ws - divm(z.ws, W.ms) * W.d.spuck;
                if (so < W.S)
                    atomicAdd(&W.occ[so * W.d.spuck + tt], -1);
                if (sn < W.S)
                    atomicAdd(&W.occ[sn * W.d.spuck + tt], 1);
            }
            wave_sync();
            if (ci == nchp - 1)
                break;
            fz_load<FORM>(recs, pick * nch + ci + 1, lane, q);
            finish();
        }
        if (MODE == FZ_MSD && kp.acf_pa && lane == 0)
            acf_after(kp, r);
        if (FORM == FZ_M && bail)
            break;
        k += 1;
        PH_MARK(W, 2);
    }
    if (moves && mv.ev_n > 0 && lane == 0)
        kp.msd_evn[r] = mv.ev;
    const FzCold kc = fz_cold();
    double dt_last = k > 0 ? (FORM == FZ_M ? dt_done : cmlog / ctotal) : kc->kdt[r];
    long long drawn = k;
    if (__ballot(F.err)) {
        st = LI ? ST_DEL_ABSENT : ST_CORRUPT;
    } else if (k < n && !bail) {
        st = ST_ABSORBING;
        if (total > 0.0) {               // only a corrupted database gets here
            st = ST_CORRUPT;
            drawn += 1;
            dt_last = readlane_d(lmlog, (int)k & 63) / total;
            t = t + dt_last;
            integ = integ + ((double)nrx * rate) * dt_last;
        }
    }
    W.nr[0] = nr;
    W.integ[0] = integ;
    steps_end<1, BITS, true>(W, kp, r, rslot, t, dt_last, kc->kstep[r] + drawn, kc->rngctr[r] + drawn, st, k);
}

template <int BITS, int FORM, int MODE>
__global__ __launch_bounds__(64 * MAX_WPG) __attribute__((amdgpu_waves_per_eu(4))) void kmc_steps_kernel_fz(KParams kp)
{
    extern __shared__ __align__(16) unsigned char smem[];
    fused_loop<BITS, FORM, MODE>(kp, smem);
}
