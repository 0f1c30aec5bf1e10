// kmcg_otf.hip -- the otf backend: per-site rates from the local environment.
//
// Included by kmcg_engine.hip (one translation unit: it shares the error
// helpers and the uniform stream).  The reference's otf step loop
// (kmos/fortran_src/base_otf.f90, the generated proclist of
// kmos/io/__init__.py:2657-3723) keeps, per process, a list of the cells
// where it can run (avail_sites) and each entry's own rate
// (rates_matrix); every step re-sums every list in list order
// (update_accum_rate, base_otf.f90:687-717), picks a process by interval
// search over the process sums and a cell by interval search over the
// running sum of the chosen list (determine_procsite, 1213-1278), then
// runs the process: deletes, lattice writes, rate updates of processes
// with a bystander on a changed site, and adds with the new rates.
//
// Layout.  One wavefront per replica, lane q owns process q (at most 64
// processes).  The lattice sits in LDS as one byte per site.  In HBM, per
// replica and process, four rows of C entries (C = cells): the list
// (cell + 1, 0 = empty), the inverse index (list position + 1 by cell),
// the entry rates and, after every 16th entry, their running sum in list
// order.  The running sum is what makes the step exact and cheap: the
// reference's full re-summation in list order equals the stored running sum
// as long as every entry from the first changed position on is re-added, so
// a step re-adds only the blocks from the smallest list position it changed
// on (sequential, in the same order as the reference's loop).  The site
// search reads those sums, then the 16 entries behind the one it finds.
//
// Rates.  gr_<proc>(cell) depends only on the bystander counts; the host
// evaluates each process's expression for every count combination once per
// parameter set (Fortran kinds: see kmos_amd/otf.py) and the kernel reads
// table[base + sum of per-bystander strides].
namespace {

constexpr int OTF_MAX_P = 64;
constexpr int OTF_MAX_V = 65536;     // sites per replica (one byte each in LDS)
constexpr int OTF_LDS = 65536;       // LDS bytes a replica's wavefront may use

// The device program, compact int32 words (built by otf_build):
//   [0, spuck)        site defaults
//   owner [P][P]      run_proc_<p>'s ops for process q: off | n_del << 16 | n_rest << 24
//   writes [P]        off | count << 16 -> 2 words per write: packed site, old | new << 16
//   byst [P]          off | count << 16 -> per bystander: packed site, then S strides
//   tbase [P]         first table entry of process q
//   touch [P]         off | count << 16 -> touchup_cell's add ops of process q
// op word:   kind (2 bits: 0 del, 2 update, 3 add) | dx, dy, dz (8 bits each) << 2, 10, 18
//            | ncond << 26 (adds)
// cond word: dx, dy, dz (7 bits each) | site - 1 (5 bits) << 21 | species << 26
// site word: dx, dy, dz (8 bits each) | site - 1 << 24
struct OtfParams {
    int P, S, spuck, T, W;
    const int *prog;                 // global copy of the program (W words)
    int off_owner, off_writes, off_byst, off_tbase, off_touch;
    int tab_lds;                     // 1: the replica's rate table is staged in LDS too
    const int *fast;                 // otf_fast_kernel: its LDS words (FW), then the op records
    int FW, off_fw, off_fb, off_ft;  // writes, bystanders, table bases within the LDS words
    const int *dims;                 // [n][4]: X, Y, Z, C
    const long long *lat_off;        // [n]: first site of the replica in `lat`
    const long long *list_off;       // [n]: first entry of the replica's rows (of otf_row(C) entries each)
    signed char *lat;
    int *sites, *back;
    double *rm, *pre;
    int *nsites;                     // [n][P]
    long long *procstat;             // [n][P]
    double *integ, *accum, *runsum;  // [n][P]
    double *table;                   // [n][T]
    double *kmc_time, *kmc_time_step;
    long long *kmc_step;
    unsigned long long *ctr;
    const unsigned *seed, *stream;
    int *status;
    const int *rep_ids;
    long long steps;
    int mode;
    // the replicas' read-back words in pinned host memory, written by every
    // kernel that changes them: OTF_OUT(P) words of 8 bytes each (integ[P],
    // accum[P], procstat[P], list sizes[P], kmc_time, kmc_time_step, kmc_step,
    // status)
    double *out;
};
constexpr int OTF_OUT(int P) { return 4 * P + 4; }

__device__ __forceinline__ int otf_wrap(int a, int n) { return a < 0 ? a + n : (a >= n ? a - n : a); }
__device__ __forceinline__ int sx8(int w, int sh) { return (int)(signed char)((w >> sh) & 0xFF); }
__device__ __forceinline__ int sx7(int w, int sh) { return (((w >> sh) & 0x7F) ^ 0x40) - 0x40; }

// The read-back words of replica r from its owner lanes (act: lane < P).
__device__ __forceinline__ void otf_export(const OtfParams &p, int r, int lane, bool act, double integ, double accum,
                                           long long pstat, int n)
{
    double *o = p.out + (long long)r * (4 * p.P + 4);
    if (act) {
        o[lane] = integ;
        o[p.P + lane] = accum;
        ((long long *)o)[2 * p.P + lane] = pstat;
        ((long long *)o)[3 * p.P + lane] = n;
    }
}
__device__ __forceinline__ void otf_export_clock(const OtfParams &p, int r, double t, double dt, long long step, int st)
{
    double *o = p.out + (long long)r * (4 * p.P + 4) + 4 * p.P;
    o[0] = t;
    o[1] = dt;
    ((long long *)o)[2] = step;
    ((long long *)o)[3] = st;
}

struct OtfCell {
    int X, Y, Z, C;
    __device__ __forceinline__ int idx(int x, int y, int z) const { return x + X * (y + Y * z); }
    __device__ __forceinline__ void xyz(int c, int &x, int &y, int &z) const
    {
        x = c % X;
        const int yz = c / X;
        y = yz % Y;
        z = yz / Y;
    }
    // the cell at (x, y, z) + (dx, dy, dz), each offset at most one period
    __device__ __forceinline__ int at(int x, int y, int z, int dx, int dy, int dz) const
    {
        return idx(otf_wrap(x + dx, X), otf_wrap(y + dy, Y), otf_wrap(z + dz, Z));
    }
};

// gr_<q>(cell): the table entry of the bystander counts around (x, y, z)
__device__ __forceinline__ double otf_gr(const int *prog, const OtfParams &p, const OtfCell &g,
                                         const signed char *slat, const double *tab, int q, int x, int y, int z)
{
    const int bt = prog[p.off_byst + q];
    const int *b = prog + (bt & 0xFFFF);
    const int nb = bt >> 16;
    int idx = 0;
    for (int k = 0; k < nb; ++k, b += 1 + p.S) {
        const int w = b[0];
        const int c = g.at(x, y, z, sx8(w, 0), sx8(w, 8), sx8(w, 16));
        const int sp = slat[p.spuck * c + ((w >> 24) & 0xFF)];
        if (sp >= 0 && sp < p.S)
            idx += b[1 + sp];
    }
    return tab[prog[p.off_tbase + q] + idx];
}

// del_proc (base_otf.f90:221-282) on the owner lane's rows: the last entry
// moves into the freed position.  Returns the first list position whose
// rate changed (the freed one, or the new end when the moved entry carries
// the same rate, so that the running sums below it stand), -1 when the
// inverse index points outside the list.
__device__ __forceinline__ int otf_del(int *srow, int *brow, double *rrow, int &n, double &run, int c)
{
    const int pos = brow[c] - 1;
    const int last = n - 1;
    if (pos < 0 || pos > last)
        return -1;
    const double gone = rrow[pos];
    run = run - gone;
    int changed = last;
    if (pos < last) {
        const int mv = srow[last];
        const double mr = rrow[last];
        srow[pos] = mv;
        rrow[pos] = mr;
        brow[mv - 1] = pos + 1;
        if (mr != gone)
            changed = pos;
    }
    srow[last] = 0;
    rrow[last] = 0.0;
    brow[c] = 0;
    n = last;
    return changed;
}

// entries from one row to the next: whole checkpoint blocks
constexpr int OTF_BLK = 16;
__host__ __device__ inline long long otf_row(int C) { return (C + OTF_BLK - 1) & ~(long long)(OTF_BLK - 1); }

// A row's running sum in list order (update_accum_rate, base_otf.f90:
// 687-717), kept after every 16th entry only: chk[j] is the sum of the first
// 16 (j + 1) entries.  Re-adds the entries from the block of position `from`
// on and returns the row's total.  Every lane walks its own row: an entry is
// one dependent addition, half a load and a sixteenth of a store, where rows
// of 16 lanes shifting a carry spent three instructions and a hazard per
// entry on four rows at a time.  Entries past the end are zero (adding zero
// changes no bit).  AHEAD blocks are on their way at a time.
template <int AHEAD>
__device__ __forceinline__ double otf_resum(const double *rrow, double *chk, int from, int n)
{
    const int b0 = from >> 4, nb = (n + OTF_BLK - 1) >> 4;
    double a = b0 > 0 ? chk[b0 - 1] : 0.0;
    if (b0 >= nb)
        return a;
    typedef double double2w __attribute__((ext_vector_type(2), aligned(8)));
    double2w v[AHEAD][8];
    auto load = [&](double2w (&w)[8], int b) {
        // past the last block: the last one again, not used
        const double2w *s = (const double2w *)(rrow + OTF_BLK * min(b, nb - 1));
#pragma unroll
        for (int k = 0; k < 8; ++k)
            w[k] = s[k];
    };
#pragma unroll
    for (int j = 0; j < AHEAD; ++j)
        load(v[j], b0 + j);
    for (int b = b0;;) {
#pragma unroll
        for (int j = 0; j < AHEAD; ++j) {
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                a = a + v[j][k].x;
                a = a + v[j][k].y;
            }
            chk[b] = a;
            if (++b >= nb)
                return a;
            load(v[j], b + AHEAD - 1);
        }
    }
}

// otf_resum for all lists a step changed at once (whole wave; `want`, from,
// n, rrow and chk per owner lane).  A lane that reads its own row alone takes
// 16 of a line's 128 bytes at a time, and with ten rows and five blocks ahead
// in eight waves per CU the lines outgrow the L1 cache: 35,000 to 50,000
// cycles of a full chip's step against 16,000 on an empty one.  Here 16
// lanes read a row's block (one line), four rows per load, OTF_DEEP blocks
// ahead in registers; each block passes through LDS to the lane that adds
// it up: 25,000 to 37,000 cycles on a full chip (33 -> 24 us per step), bound
// by its additions and their LDS reads.  Up to OTF_ROWS lists at a time.
// Returns the row's total where `want`.
constexpr int OTF_ROWS = 12, OTF_DEEP = 6, OTF_STAGE = OTF_BLK + 2;   // (16-byte aligned, spread over the banks)

__device__ __forceinline__ double otf_resum_wave(const double *rm, double *pre, long long crow, int P, bool want,
                                                 int from, int n, double tot, double *stage, int *ids, int lane)
{
    constexpr int SETS = OTF_ROWS / 4;
    const int b0 = from >> 4, nb = (n + OTF_BLK - 1) >> 4;
    // short tails only (rates that do not differ within a list): each lane
    // its own
    if (!__ballot(want && nb - b0 > 2))
        return want ? otf_resum<2>(rm + lane * crow, pre + lane * (crow / OTF_BLK), from, n) : tot;
    // the checkpoints through a buffer descriptor: lanes past their last
    // block store outside it, without a branch
    typedef int int2v __attribute__((ext_vector_type(2)));
    const int crow_chk = (int)(crow / OTF_BLK);
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(pre, 0, P * crow_chk * 8, 0x00027000);
    const double *chk = pre + (want ? lane : 0) * crow_chk;
    const unsigned at0 = (unsigned)((want ? lane : 0) * crow_chk + b0) * 8u;
    double a = want && b0 > 0 ? chk[b0 - 1] : 0.0;
    unsigned long long todo = __ballot(want && b0 < nb);
    while (todo) {
        // this group's lists: the first OTF_ROWS pending lanes
        const int rank = __popcll(todo & ((1ull << lane) - 1ull));
        const bool mine = ((todo >> lane) & 1) && rank < OTF_ROWS;
        if (lane < OTF_ROWS)
            ids[lane] = -1;
        wave_sync();
        if (mine)
            ids[rank] = lane;
        wave_sync();
        const char *rows = (const char *)rm;             // (a replica's rows: below 4 GiB)
        unsigned src[SETS];
        int last[SETS];
#pragma unroll
        for (int i = 0; i < SETS; ++i) {
            const int id = ids[4 * i + (lane >> 4)];
            const int f = __builtin_amdgcn_ds_bpermute(id << 2, b0), e = __builtin_amdgcn_ds_bpermute(id << 2, nb);
            // (behind its last block a row reads that one again, unused)
            last[i] = id >= 0 ? e - f - 1 : 0;
            src[i] = (unsigned)(max(id, 0) * (int)crow + (id >= 0 ? OTF_BLK * f : 0) + (lane & 15)) * 8u;
        }
        const int T = mine ? nb - b0 : 0;
        double v[OTF_DEEP][SETS];
#pragma unroll
        for (int j = 0; j < OTF_DEEP; ++j)
#pragma unroll
            for (int i = 0; i < SETS; ++i)
                v[j][i] = *(const double *)(rows + (src[i] + 8u * OTF_BLK * (unsigned)min(j, last[i])));
        const double *my = stage + (mine ? rank : 0) * OTF_STAGE;
        double sum = a;
        for (int t0 = 0; __ballot(t0 < T); t0 += OTF_DEEP) {
#pragma unroll
            for (int j = 0; j < OTF_DEEP; ++j) {
                const int t = t0 + j;
#pragma unroll
                for (int i = 0; i < SETS; ++i) {
                    stage[(4 * i + (lane >> 4)) * OTF_STAGE + (lane & 15)] = v[j][i];
                    v[j][i] = *(const double *)(rows +
                                                (src[i] + 8u * OTF_BLK * (unsigned)min(t + OTF_DEEP, last[i])));
                }
                wave_sync();
                double w[OTF_BLK];
#pragma unroll
                for (int k = 0; k < OTF_BLK; ++k)
                    w[k] = my[k];
#pragma unroll
                for (int k = 0; k < OTF_BLK; ++k)
                    sum = sum + w[k];
                union {
                    double d;
                    int2v v;
                } out;
                out.d = sum;
                __builtin_amdgcn_raw_buffer_store_b64(out.v, rs, t < T ? at0 + 8u * (unsigned)t : FZ_NONE, 0, 0);
                a = t < T ? sum : a;
                wave_sync();
            }
        }
        todo &= ~__ballot(mine);
    }
    return want ? a : tot;
}

// The running sum of the first pos + 1 entries of a row.
__device__ __forceinline__ double otf_prefix(const double *rrow, const double *chk, int pos)
{
    double a = pos >> 4 ? chk[(pos >> 4) - 1] : 0.0;
    for (int j = pos & ~(OTF_BLK - 1); j <= pos; ++j)
        a = a + rrow[j];
    return a;
}

// The cell of the first entry of a row of np entries whose running sum
// exceeds vs (interval search of determine_procsite, base_otf.f90:1213-1278;
// past the end the last entry, walked left over equal sums).  Uniform call:
// 64-ary over the checkpoints, four of them per lane in the last round, then
// the 16 entries behind the one found, added by every lane alike, their
// cells read along with them.
__device__ __forceinline__ int otf_pick(const int *srow, const double *rrow, const double *chk, int np, double vs,
                                        int lane)
{
    int lo = 0, hi = np >> 4;
    while (hi - lo > 256) {
        const int stride = (hi - lo + 63) >> 6;
        const int at = lo + (lane + 1) * stride - 1;
        const bool in = at < hi;
        const double pv = in ? chk[at] : 0.0;
        const unsigned long long mm = __ballot(in && pv > vs);
        if (mm) {
            const int k = __ffsll((long long)mm) - 1;
            hi = lo + (k + 1) * stride - 1;
            lo = lo + k * stride;
        } else {
            lo = lo + (int)__popcll(__ballot(in)) * stride;
        }
    }
    double c4[4];
#pragma unroll
    for (int k = 0; k < 4; ++k)
        c4[k] = lo + 4 * lane + k < hi ? chk[lo + 4 * lane + k] : 0.0;
    int mine = 4;
#pragma unroll
    for (int k = 3; k >= 0; --k)
        mine = lo + 4 * lane + k < hi && c4[k] > vs ? k : mine;
    const unsigned long long mc = __ballot(mine < 4);
    const int l0 = mc ? __ffsll((long long)mc) - 1 : 0;
    const int blk = mc ? lo + 4 * l0 + readlane_i(mine, l0) : hi;
    double a = blk > 0 ? chk[blk - 1] : 0.0;
    const int mycell = lane < OTF_BLK && OTF_BLK * blk + lane < np ? srow[OTF_BLK * blk + lane] : 0;
    double e[OTF_BLK];
#pragma unroll
    for (int k = 0; k < OTF_BLK; ++k)
        e[k] = OTF_BLK * blk + k < np ? rrow[OTF_BLK * blk + k] : 0.0;
    int at = 0;
#pragma unroll
    for (int k = 0; k < OTF_BLK; ++k) {
        a = a + e[k];
        at += a > vs ? 0 : 1;
    }
    at = __builtin_amdgcn_readfirstlane(at);
    if (OTF_BLK * blk + at < np)
        return readlane_i(mycell, at) - 1;
    int pos = np - 1;
    while (pos > 0 && otf_prefix(rrow, chk, pos - 1) >= otf_prefix(rrow, chk, pos))
        --pos;
    return __builtin_amdgcn_readfirstlane(srow[pos]) - 1;
}

__device__ __forceinline__ bool otf_conds(const OtfParams &p, const OtfCell &g, const signed char *slat,
                                          const int *cd, int ncond, int x, int y, int z)
{
    for (int j = 0; j < ncond; ++j) {
        const int w = cd[j];
        const int c = g.at(x, y, z, sx7(w, 0), sx7(w, 7), sx7(w, 14));
        if (slat[p.spuck * c + ((w >> 21) & 0x1F)] != ((w >> 26) & 0x3F))
            return false;
    }
    return true;
}

// MODE 0: initialize_state (default species everywhere, touchup_cell over
// the cells with x fastest); MODE 1: _adjust_database after a new lattice
// (touchup_cell with x outermost: delete the cell's entry, then add it if
// the conditions hold); MODE 2: recalculate_rates_matrix (every listed
// entry takes its cell's rate under new parameters).  Each ends with the
// rows' running sums.  The program and tables are read from global memory
// (a one-off pass).
__global__ __launch_bounds__(64) void otf_setup_kernel(OtfParams p)
{
    extern __shared__ signed char slat[];
    const int r = p.rep_ids[blockIdx.x];
    const int lane = threadIdx.x;
    const OtfCell g{p.dims[4 * r], p.dims[4 * r + 1], p.dims[4 * r + 2], p.dims[4 * r + 3]};
    const int V = g.C * p.spuck;
    const int *prog = p.prog;
    signed char *glat = p.lat + p.lat_off[r];
    if (p.mode == 0) {
        for (int i = lane; i < V; i += 64)
            glat[i] = (signed char)prog[i % p.spuck];     // site defaults head the program
        __syncthreads();
    }
    for (int i = lane; i < V; i += 64)
        slat[i] = glat[i];
    __syncthreads();
    if (lane >= p.P)
        return;
    const int q = lane;
    const long long lo = p.list_off[r] + q * otf_row(g.C);
    int *srow = p.sites + lo;
    int *brow = p.back + lo;
    double *rrow = p.rm + lo;
    double *prow = p.pre + lo / OTF_BLK;
    const double *tab = p.table + (long long)r * p.T;
    const int slot = r * p.P + q;
    int n = p.nsites[slot];
    double run = p.runsum[slot];
    if (p.mode == 0) {
        for (int c = 0; c < g.C; ++c) {
            srow[c] = 0;
            brow[c] = 0;
            rrow[c] = 0.0;
        }
        n = 0;
        run = 0.0;
    }
    if (p.mode == 2) {
        for (int j = 0; j < n; ++j) {
            if (srow[j] < 1 || srow[j] > g.C)
                continue;
            int x, y, z;
            g.xyz(srow[j] - 1, x, y, z);
            rrow[j] = otf_gr(prog, p, g, slat, tab, q, x, y, z);
        }
        // reaccumulate_rates_matrix (base_otf.f90:366-387): memory order
        run = 0.0;
        for (int j = 0; j < n; ++j)
            run = run + rrow[j];
    } else {
        const int tt = prog[p.off_touch + q];
        for (int k = 0; k < g.C; ++k) {
            int x, y, z;
            if (p.mode == 0) {
                g.xyz(k, x, y, z);
            } else {
                // x outermost, then y, then z
                z = k % g.Z;
                const int xy = k / g.Z;
                y = xy % g.Y;
                x = xy / g.Y;
            }
            const int c = g.idx(x, y, z);
            if (p.mode == 1 && brow[c] && otf_del(srow, brow, rrow, n, run, c) < 0) {
                p.status[r] = KMCG_REPLICA_CORRUPT;
                break;
            }
            const int *op = prog + (tt & 0xFFFF);
            for (int m = 0; m < (tt >> 16); ++m) {
                const int ncond = (op[0] >> 26) & 0x3F;
                if (otf_conds(p, g, slat, op + 1, ncond, x, y, z) && n < g.C) {
                    const double rate = otf_gr(prog, p, g, slat, tab, q, x, y, z);
                    srow[n] = c + 1;
                    brow[c] = n + 1;
                    rrow[n] = rate;
                    run = run + rate;
                    n += 1;
                }
                op += 1 + ncond;
            }
        }
    }
    otf_resum<5>(rrow, prow, 0, n);
    p.nsites[slot] = n;
    p.runsum[slot] = run;
    if (p.mode == 0) {
        p.procstat[slot] = 0;
        p.integ[slot] = 0.0;
        p.accum[slot] = 0.0;
        if (q == 0) {
            p.kmc_time[r] = 0.0;
            p.kmc_time_step[r] = 0.0;
            p.kmc_step[r] = 0;
            p.ctr[r] = 0;
            p.status[r] = KMCG_REPLICA_OK;
        }
    }
    otf_export(p, r, lane, true, p.integ[slot], p.accum[slot], p.procstat[slot], n);
    wave_sync();
    if (q == 0)
        otf_export_clock(p, r, p.kmc_time[r], p.kmc_time_step[r], p.kmc_step[r], p.status[r]);
}

// do_kmc_steps for `steps` steps (fewer when the replica stops).  LDS holds
// the program, the replica's rate table (TLDS) and its lattice.
template <bool TLDS>
__global__ __launch_bounds__(64) void otf_steps_kernel(OtfParams p)
{
    extern __shared__ __align__(16) int otf_smem[];
    const int r = p.rep_ids[blockIdx.x];
    const int lane = threadIdx.x;
    const int P = p.P;
    const OtfCell g{p.dims[4 * r], p.dims[4 * r + 1], p.dims[4 * r + 2], p.dims[4 * r + 3]};
    const int V = g.C * p.spuck;
    int *prog = otf_smem;
    const int W2 = (p.W + 1) & ~1;
    double *stab = reinterpret_cast<double *>(otf_smem + W2);
    signed char *slat = reinterpret_cast<signed char *>(otf_smem + W2 + (TLDS ? 2 * p.T : 0));
    signed char *glat = p.lat + p.lat_off[r];
    for (int i = lane; i < p.W; i += 64)
        prog[i] = p.prog[i];
    if (TLDS)
        for (int i = lane; i < p.T; i += 64)
            stab[i] = p.table[(long long)r * p.T + i];
    for (int i = lane; i < V; i += 64)
        slat[i] = glat[i];
    __syncthreads();
    const double *tab = TLDS ? stab : p.table + (long long)r * p.T;
    int st = p.status[r];
    if (st != KMCG_REPLICA_OK)
        return;
    const bool act = lane < P;
    const int q = act ? lane : 0;
    const long long base = p.list_off[r];
    const long long crow = otf_row(g.C);
    const long long lo = base + q * crow;
    int *srow = p.sites + lo;
    int *brow = p.back + lo;
    double *rrow = p.rm + lo;
    double *chk = p.pre + lo / OTF_BLK;
    const int slot = r * P + q;
    int n = act ? p.nsites[slot] : 0;
    double tot = (act && n > 0) ? otf_prefix(rrow, chk, n - 1) : 0.0;
    double integ = act ? p.integ[slot] : 0.0;
    double run = act ? p.runsum[slot] : 0.0;
    double my_acc = act ? p.accum[slot] : 0.0;
    long long pstat = act ? p.procstat[slot] : 0;
    double t = p.kmc_time[r];
    double t_step = p.kmc_time_step[r];
    long long kstep = p.kmc_step[r];
    unsigned long long ctr = p.ctr[r];
    const unsigned seed = p.seed[r], stream = p.stream[r];
    const unsigned long long ctr0 = ctr;
    double lmlog = 0.0, lu1 = 0.0, lu2 = 0.0;
    for (long long s = 0; s < p.steps; ++s) {
        // uniforms of 64 steps at a time: lane i draws step s + i
        const int uj = (int)s & 63;
        if (uj == 0) {
            const FzUni un = fz_uniforms(seed, stream, ctr0 + (unsigned long long)s + lane);
            lmlog = un.mlog;
            lu1 = un.u1;
            lu2 = un.u2;
        }
        // update_accum_rate: accum(i) = accum(i-1) + sum of list i
        double acc = 0.0;
        for (int i = 0; i < P; ++i) {
            const double ti = readlane_d(tot, i);
            acc = i == 0 ? ti : acc + ti;
            if (lane == i)
                my_acc = acc;
        }
        run = tot;
        const double total = acc;
        if (!(total > 0.0)) {
            st = KMCG_REPLICA_ABSORBING;
            break;
        }
        ctr += 1;
        // update_clocks, update_integ_rate
        const double dt = readlane_d(lmlog, uj) / total;
        t_step = dt;
        t = t + dt;
        kstep += 1;
        integ = integ + tot * dt;
        // determine_procsite: the first process whose accum exceeds the
        // value (interval_search_real); past the end, the last one, walked
        // left over equal sums
        const double v = readlane_d(lu1, uj) * total;
        const unsigned long long mp = __ballot(act && my_acc > v);
        int proc = mp ? __ffsll((long long)mp) - 1 : P - 1;
        if (!mp)
            while (proc > 0 && readlane_d(my_acc, proc - 1) >= readlane_d(my_acc, proc))
                --proc;
        const int np = readlane_i(n, proc);
        const double vs = readlane_d(lu2, uj) * readlane_d(tot, proc);
        const int cell = otf_pick(p.sites + base + proc * crow, p.rm + base + proc * crow,
                                  p.pre + (base + proc * crow) / OTF_BLK, np, vs, lane);
        int x, y, z;
        g.xyz(cell, x, y, z);
        if (lane == proc)
            pstat += 1;
        // run_proc_<proc>: the owner lane's deletes
        int dirty = 0x7fffffff;
        bool corrupt = false;
        const int own = prog[p.off_owner + proc * P + q];
        const int *w = prog + (own & 0xFFFF);
        const int nd = act ? (own >> 16) & 0xFF : 0;
        const int nrest = act ? (own >> 24) & 0xFF : 0;
        for (int k = 0; k < nd; ++k, ++w) {
            const int c = g.at(x, y, z, sx8(w[0], 2), sx8(w[0], 10), sx8(w[0], 18));
            if (brow[c]) {
                const int d = otf_del(srow, brow, rrow, n, run, c);
                if (d < 0)
                    corrupt = true;
                else
                    dirty = min(dirty, d);
            }
        }
        // lattice writes
        const int wt = prog[p.off_writes + proc];
        bool bad = false;
        if (lane < (wt >> 16)) {
            const int *ww = prog + (wt & 0xFFFF) + 2 * lane;
            const int c = g.at(x, y, z, sx8(ww[0], 0), sx8(ww[0], 8), sx8(ww[0], 16));
            const int site = p.spuck * c + ((ww[0] >> 24) & 0xFF);
            bad = slat[site] != (ww[1] & 0xFFFF);
            slat[site] = (signed char)(ww[1] >> 16);
        }
        __syncthreads();
        // the owner lane's rate updates, which come before its adds: in
        // batches of up to eight, their inverse indices read together, then
        // their old rates, then the new ones applied in program order
        int k = 0;
        for (;;) {
            int m = 0;
            while (m < 8 && k + m < nrest && (w[m] & 3) == 2)
                ++m;
            if (m == 0)
                break;
            int cx8[8], cy8[8], cz8[8], c8[8], bk8[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                if (j < m) {
                    cx8[j] = otf_wrap(x + sx8(w[j], 2), g.X);
                    cy8[j] = otf_wrap(y + sx8(w[j], 10), g.Y);
                    cz8[j] = otf_wrap(z + sx8(w[j], 18), g.Z);
                    c8[j] = g.idx(cx8[j], cy8[j], cz8[j]);
                    bk8[j] = brow[c8[j]];
                }
            }
            double old8[8], new8[8];
#pragma unroll
            for (int j = 0; j < 8; ++j)
                if (j < m && bk8[j] > 0 && bk8[j] <= n)
                    old8[j] = rrow[bk8[j] - 1];
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                if (j < m) {
                    if (bk8[j] > n) {
                        corrupt = true;
                    } else if (bk8[j]) {
                        const int at = bk8[j] - 1;
                        double old = old8[j];
#pragma unroll
                        for (int j2 = 0; j2 < j; ++j2)       // the same cell twice in one batch
                            if (c8[j2] == c8[j] && bk8[j2] == bk8[j])
                                old = new8[j2];
                        new8[j] = otf_gr(prog, p, g, slat, tab, q, cx8[j], cy8[j], cz8[j]);
                        run = run + new8[j] - old;
                        rrow[at] = new8[j];
                        if (new8[j] != old)
                            dirty = min(dirty, at);
                    }
                }
            }
            w += m;
            k += m;
        }
        // then its adds, in program order
        for (; k < nrest; ++k) {
            const int op = w[0];
            const int cx = otf_wrap(x + sx8(op, 2), g.X), cy = otf_wrap(y + sx8(op, 10), g.Y),
                      cz = otf_wrap(z + sx8(op, 18), g.Z);
            const int c = g.idx(cx, cy, cz);
            if ((op & 3) == 2) {
                if (brow[c] > n) {
                    corrupt = true;
                } else if (brow[c]) {
                    const int at = brow[c] - 1;
                    const double rate = otf_gr(prog, p, g, slat, tab, q, cx, cy, cz);
                    const double old = rrow[at];
                    run = run + rate - old;
                    rrow[at] = rate;
                    if (rate != old)
                        dirty = min(dirty, at);
                }
                w += 1;
            } else {
                const int ncond = (op >> 26) & 0x3F;
                if (n >= g.C) {
                    corrupt = true;             // an add to a full list
                } else if (otf_conds(p, g, slat, w + 1, ncond, x, y, z)) {
                    const double rate = otf_gr(prog, p, g, slat, tab, q, cx, cy, cz);
                    srow[n] = c + 1;
                    brow[c] = n + 1;
                    rrow[n] = rate;
                    run = run + rate;
                    dirty = min(dirty, n);
                    n += 1;
                }
                w += 1 + ncond;
            }
        }
        // (an entry deleted at the end leaves its block's checkpoint behind
        // the last whole block: not read)
        if (act && dirty != 0x7fffffff)
            tot = otf_resum<5>(rrow, chk, min(dirty, n), n);
        if (__ballot(bad)) {
            st = KMCG_REPLICA_SPECIES_MISMATCH;
            break;
        }
        if (__ballot(corrupt)) {
            st = KMCG_REPLICA_CORRUPT;
            break;
        }
    }
    __syncthreads();
    for (int i = lane; i < V; i += 64)
        glat[i] = slat[i];
    if (act) {
        p.nsites[slot] = n;
        p.procstat[slot] = pstat;
        p.integ[slot] = integ;
        p.accum[slot] = my_acc;
        p.runsum[slot] = run;
    }
    otf_export(p, r, lane, act, integ, my_acc, pstat, n);
    if (lane == 0) {
        otf_export_clock(p, r, t, t_step, kstep, st);
        p.kmc_time[r] = t;
        p.kmc_time_step[r] = t_step;
        p.kmc_step[r] = kstep;
        p.ctr[r] = ctr;
        p.status[r] = st;
    }
}

// The step loop with one lane per list operation (for the models that
// otf_build_fast takes and the lattices that otf_launch finds large enough;
// the others run otf_steps_kernel).
//
// A step of the intZGB model has 13 to 23 deletes, 40 to 62 rate updates and
// 5 to 13 adds on ten lists.  An owner lane that walks its own ones waits for
// two or three dependent reads per operation and looks its bystanders up one
// by one (40,000 of a step's 80,000 cycles).  Here every operation of the
// executed process is a lane (two rounds of 64): inverse index, old rate,
// conditions and new rate of all of them are found at once, and the owner
// lanes only apply what takes place, in the reference's order, from LDS.
// Deletes precede updates and adds and name each (process, cell) once, so an
// entry's place changes only by the moves of the deletes, which stay in
// registers.
//
// Op records of an executed process (global memory, read while its cell is
// searched): 64 owner words: first op | ops << 8 | deletes << 16 | updates << 24;
// then 128 pairs: kind (0 delete, 1 none, 2 update, 3 add) | process << 2 |
// same cell updated before << 8 | conditions << 9 | their LDS word << 16;
// dx, dy, dz (8 bits each).
constexpr int OTF_OPS = 128;
constexpr int OTF_FREC = 64 + 2 * OTF_OPS;

__global__ __launch_bounds__(64) void otf_fast_kernel(OtfParams p)
{
    extern __shared__ __align__(16) int otf_smem[];
    const int r = p.rep_ids[blockIdx.x];
    const int lane = threadIdx.x;
    const int P = p.P;
    const OtfCell g{p.dims[4 * r], p.dims[4 * r + 1], p.dims[4 * r + 2], p.dims[4 * r + 3]};
    const int V = g.C * p.spuck;
    // LDS: program words, rate table, the operations' results, lattice
    int *prog = otf_smem;
    double *tab = reinterpret_cast<double *>(otf_smem + ((p.FW + 1) & ~1));
    double *eold = tab + p.T, *enew = eold + OTF_OPS;
    int *ecell = reinterpret_cast<int *>(enew + OTF_OPS), *eback = ecell + OTF_OPS;
    signed char *slat = reinterpret_cast<signed char *>(eback + OTF_OPS);
    signed char *glat = p.lat + p.lat_off[r];
    for (int i = lane; i < p.FW; i += 64)
        prog[i] = p.fast[i];
    for (int i = lane; i < p.T; i += 64)
        tab[i] = p.table[(long long)r * p.T + i];
    for (int i = lane; i < V; i += 64)
        slat[i] = glat[i];
    __syncthreads();
    int st = p.status[r];
    if (st != KMCG_REPLICA_OK)
        return;
    const int *recs = p.fast + p.FW;
    const bool act = lane < P;
    const int q = act ? lane : 0;
    const long long base = p.list_off[r], crow = otf_row(g.C);
    const long long lo = base + q * crow;
    int *srow = p.sites + lo;
    int *brow = p.back + lo;
    double *rrow = p.rm + lo;
    double *chk = p.pre + lo / OTF_BLK;
    const int slot = r * P + q;
    int n = act ? p.nsites[slot] : 0;
    double tot = (act && n > 0) ? otf_prefix(rrow, chk, n - 1) : 0.0;
    double integ = act ? p.integ[slot] : 0.0;
    double run = act ? p.runsum[slot] : 0.0;
    double my_acc = act ? p.accum[slot] : 0.0;
    long long pstat = act ? p.procstat[slot] : 0;
    double t = p.kmc_time[r];
    double t_step = p.kmc_time_step[r];
    const long long kstep0 = p.kmc_step[r];
    const unsigned long long ctr0 = p.ctr[r];
    const unsigned seed = p.seed[r], stream = p.stream[r];
    double lmlog = 0.0, lu1 = 0.0, lu2 = 0.0;
    long long s = 0;
    for (; s < p.steps; ++s) {
        // uniforms of 64 steps at a time: lane i draws step s + i
        const int uj = (int)s & 63;
        if (uj == 0) {
            const FzUni un = fz_uniforms(seed, stream, ctr0 + (unsigned long long)s + lane);
            lmlog = un.mlog;
            lu1 = un.u1;
            lu2 = un.u2;
        }
        // update_accum_rate: accum(i) = accum(i-1) + sum of list i
        double acc = 0.0;
        for (int i = 0; i < P; ++i) {
            const double ti = readlane_d(tot, i);
            acc = i == 0 ? ti : acc + ti;
            if (lane == i)
                my_acc = acc;
        }
        run = tot;
        const double total = acc;
        if (!(total > 0.0)) {
            st = KMCG_REPLICA_ABSORBING;
            break;
        }
        // update_clocks, update_integ_rate
        const double dt = readlane_d(lmlog, uj) / total;
        t_step = dt;
        t = t + dt;
        integ = integ + tot * dt;
        // determine_procsite (the process: see otf_steps_kernel)
        const double v = readlane_d(lu1, uj) * total;
        const unsigned long long mp = __ballot(act && my_acc > v);
        int proc = mp ? __ffsll((long long)mp) - 1 : P - 1;
        if (!mp)
            while (proc > 0 && readlane_d(my_acc, proc - 1) >= readlane_d(my_acc, proc))
                --proc;
        // its records are on their way during the search
        const int *rec = recs + proc * OTF_FREC;
        const int own = rec[lane];
        const int2 op0 = ((const int2 *)(rec + 64))[lane], op1 = ((const int2 *)(rec + 64))[64 + lane];
        const int np = readlane_i(n, proc);
        const double vs = readlane_d(lu2, uj) * readlane_d(tot, proc);
        const int cell = otf_pick(p.sites + base + proc * crow, p.rm + base + proc * crow,
                                  p.pre + (base + proc * crow) / OTF_BLK, np, vs, lane);
        int x, y, z;
        g.xyz(cell, x, y, z);
        if (lane == proc)
            pstat += 1;
        // every operation's cell and inverse index
        int oc[2], ob[2], ocx[2], ocy[2], ocz[2], okind[2], oq[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int2 o = h ? op1 : op0;
            okind[h] = o.x & 3;
            oq[h] = (o.x >> 2) & 63;
            ocx[h] = otf_wrap(x + sx8(o.y, 0), g.X);
            ocy[h] = otf_wrap(y + sx8(o.y, 8), g.Y);
            ocz[h] = otf_wrap(z + sx8(o.y, 16), g.Z);
            oc[h] = g.idx(ocx[h], ocy[h], ocz[h]);
            ob[h] = p.back[base + oq[h] * crow + oc[h]];
        }
        // lattice writes
        const int wt = prog[p.off_fw + proc];
        bool bad = false;
        if (lane < (wt >> 16)) {
            const int *ww = prog + (wt & 0xFFFF) + 2 * lane;
            const int c = g.at(x, y, z, sx8(ww[0], 0), sx8(ww[0], 8), sx8(ww[0], 16));
            const int site = p.spuck * c + ((ww[0] >> 24) & 0xFF);
            bad = slat[site] != (ww[1] & 0xFFFF);
            slat[site] = (signed char)(ww[1] >> 16);
        }
        __syncthreads();
        // which take place, old and new rates
        bool corrupt = false;
        unsigned long long on[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int2 o = h ? op1 : op0;
            const int nq = __builtin_amdgcn_ds_bpermute(oq[h] << 2, n);
            const bool listed = okind[h] != 1 && okind[h] != 3 && ob[h] != 0;
            const bool off = listed && (ob[h] < 0 || ob[h] > nq);
            corrupt = corrupt || off;
            bool take = listed && !off;
            double old = 0.0, rate = 0.0;
            if (take)
                old = p.rm[base + oq[h] * crow + ob[h] - 1];
            if (okind[h] == 3)
                take = otf_conds(p, g, slat, prog + (int)((unsigned)o.x >> 16), (o.x >> 9) & 0x3F, x, y, z);
            if (take && okind[h] >= 2) {
                const int bt = prog[p.off_fb + oq[h]], nb = bt >> 16;
                const int *b = prog + (bt & 0xFFFF);
                int idx = prog[p.off_ft + oq[h]];
                for (int k0 = 0; k0 < nb; k0 += 4) {
                    int sw[4], sp[4];
#pragma unroll
                    for (int k = 0; k < 4; ++k)
                        sw[k] = b[min(k0 + k, nb - 1) * (1 + p.S)];
#pragma unroll
                    for (int k = 0; k < 4; ++k)
                        sp[k] = slat[p.spuck * g.at(ocx[h], ocy[h], ocz[h], sx8(sw[k], 0), sx8(sw[k], 8), sx8(sw[k], 16)) +
                                     ((sw[k] >> 24) & 0xFF)];
#pragma unroll
                    for (int k = 0; k < 4; ++k)
                        if (k0 + k < nb && sp[k] >= 0 && sp[k] < p.S)
                            idx += b[(k0 + k) * (1 + p.S) + 1 + sp[k]];
                }
                rate = tab[idx];
            }
            const int e = 64 * h + lane;
            ecell[e] = oc[h];
            eback[e] = ob[h];
            eold[e] = (o.x >> 8) & 1 ? rate : old;      // updated before in this step: its new rate
            enew[e] = rate;
            on[h] = __ballot(take);
        }
        // this owner lane's run of operations
        const int first = own & 0xFF, ndel = (own >> 16) & 0xFF, nupd = (own >> 24) & 0xFF;
        unsigned bits;
        {
            const unsigned long long l0 = on[0] >> (first & 63), l1 = on[1] >> (first & 63);
            const unsigned long long up = (first & 63) ? on[1] << (64 - (first & 63)) : 0ull;
            bits = (unsigned)(first < 64 ? l0 | up : l1);
            const int len = (own >> 8) & 0xFF;
            bits = act ? bits & ((1u << len) - 1u) : 0u;
        }
        int dirty = 0x7fffffff;
        __syncthreads();
        // deletes (del_proc, base_otf.f90:221-282): the last entry moves
        // into the freed place
        unsigned db = bits & ((1u << ndel) - 1u);
        {
            const int n0 = n, nd = __popc(db);
            int tc[4];
            double tr[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                tc[i] = i < nd && n0 - 1 - i >= 0 ? srow[n0 - 1 - i] : 0;
                tr[i] = i < nd && n0 - 1 - i >= 0 ? rrow[n0 - 1 - i] : 0.0;
            }
            int mvc[4] = {0, 0, 0, 0}, mvp[4] = {0, 0, 0, 0};
            double mvr[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if (db) {
                    const int e = first + __builtin_ctz(db);
                    db &= db - 1;
                    const int c = ecell[e];
                    int pos = eback[e] - 1;
                    const double gone = eold[e];
                    const int last = n - 1;
                    int mv = tc[i];
                    double mr = tr[i];
#pragma unroll
                    for (int j = 0; j < i; ++j) {
                        pos = mvc[j] == c + 1 ? mvp[j] : pos;
                        mr = mvc[j] && mvp[j] == last ? mvr[j] : mr;
                        mv = mvc[j] && mvp[j] == last ? mvc[j] : mv;
                    }
                    run = run - gone;
                    int changed = last;
                    if (pos < last) {
                        srow[pos] = mv;
                        rrow[pos] = mr;
                        brow[mv - 1] = pos + 1;
                        if (mr != gone)
                            changed = pos;
                        mvc[i] = mv;
                        mvp[i] = pos;
                        mvr[i] = mr;
                    }
                    srow[last] = 0;
                    rrow[last] = 0.0;
                    brow[c] = 0;
                    n = last;
                    dirty = min(dirty, changed);
                }
            }
            // rate updates, in program order
            for (unsigned ub = (bits >> ndel) & ((1u << nupd) - 1u); ub; ub &= ub - 1) {
                const int e = first + ndel + __builtin_ctz(ub);
                const int c = ecell[e];
                int pos = eback[e] - 1;
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    pos = mvc[j] == c + 1 ? mvp[j] : pos;
                const double old = eold[e], rate = enew[e];
                run = run + rate - old;
                rrow[pos] = rate;
                if (rate != old)
                    dirty = min(dirty, pos);
            }
        }
        // adds, in program order
        for (unsigned ab = bits >> (ndel + nupd); ab; ab &= ab - 1) {
            const int e = first + ndel + nupd + __builtin_ctz(ab);
            const int c = ecell[e];
            const double rate = enew[e];
            if (n >= g.C) {
                corrupt = true;             // an add to a full list
            } else {
                srow[n] = c + 1;
                brow[c] = n + 1;
                rrow[n] = rate;
                run = run + rate;
                dirty = min(dirty, n);
                n += 1;
            }
        }
        tot = otf_resum_wave(p.rm + base, p.pre + base / OTF_BLK, crow, P, act && dirty != 0x7fffffff, min(dirty, n), n,
                             tot, eold, ecell, lane);
        if (__ballot(bad)) {
            st = KMCG_REPLICA_SPECIES_MISMATCH;
            s += 1;
            break;
        }
        if (__ballot(corrupt)) {
            st = KMCG_REPLICA_CORRUPT;
            s += 1;
            break;
        }
    }
    __syncthreads();
    for (int i = lane; i < V; i += 64)
        glat[i] = slat[i];
    if (act) {
        p.nsites[slot] = n;
        p.procstat[slot] = pstat;
        p.integ[slot] = integ;
        p.accum[slot] = my_acc;
        p.runsum[slot] = run;
    }
    otf_export(p, r, lane, act, integ, my_acc, pstat, n);
    if (lane == 0) {
        otf_export_clock(p, r, t, t_step, kstep0 + s, st);
        p.kmc_time[r] = t;
        p.kmc_time_step[r] = t_step;
        p.kmc_step[r] = kstep0 + s;
        p.ctr[r] = ctr0 + (unsigned long long)s;
        p.status[r] = st;
    }
}

} // namespace

// ===========================================================================
// host side
// ===========================================================================
struct kmcg_otf_model {
    std::vector<int32_t> blob;
    int P = 0, S = 0, spuck = 0, K = 0, T = 0;
    int reach[3] = {0, 0, 0};        // largest |offset| per dimension
    std::vector<int> prog;           // the device program (see build)
    int off_owner = 0, off_writes = 0, off_byst = 0, off_tbase = 0, off_touch = 0;
    // otf_fast_kernel's words (empty: not for this model): FW LDS words, then
    // the op records; the largest offset of an operation per dimension
    std::vector<int> fast;
    int FW = 0, off_fw = 0, off_fb = 0, off_ft = 0;
    int op_reach[3] = {0, 0, 0};
};

struct kmcg_otf_batch {
    const kmcg_otf_model *m = nullptr;
    int n = 0, device = 0, maxV = 0;
    hipStream_t stream = nullptr;
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    float last_ms = 0.f;
    bool timed = false;
    std::vector<int> dims;           // [n][4]
    std::vector<long long> lat_off, list_off;
    long long lat_total = 0, list_total = 0;
    int *d_prog = nullptr, *d_dims = nullptr, *d_rep = nullptr;
    long long *d_lat_off = nullptr, *d_list_off = nullptr;
    signed char *d_lat = nullptr;
    int *d_sites = nullptr, *d_back = nullptr, *d_nsites = nullptr, *d_status = nullptr;
    double *d_rm = nullptr, *d_pre = nullptr, *d_integ = nullptr, *d_accum = nullptr, *d_runsum = nullptr;
    double *d_table = nullptr, *d_time = nullptr, *d_dt = nullptr;
    long long *d_procstat = nullptr, *d_step = nullptr;
    unsigned long long *d_ctr = nullptr;
    unsigned *d_seed = nullptr, *d_stream = nullptr;
    std::vector<double> rates, userpar;  // per replica, as last set
    double *h_out = nullptr;             // OtfParams::out
    int last_form = 0;                   // kmcg_otf_last_form
    const long long *out(int r) const { return (const long long *)h_out + (size_t)r * OTF_OUT(m->P); }
    int status(int r) const { return (int)out(r)[4 * m->P + 3]; }
};

namespace {

// x ** n for an integer n: binary powering from the low bit, 1/r for a
// negative n (the form the reference's compiler emits for real ** integer)
template <class F>
F otf_powi(F a, long long n)
{
    unsigned long long u = n < 0 ? (unsigned long long)(-n) : (unsigned long long)n;
    F r = F(1);
    while (u) {
        if (u & 1)
            r = r * a;
        u >>= 1;
        if (u)
            a = a * a;
    }
    return n < 0 ? F(1) / r : r;
}

long long otf_ipow(long long a, long long n)
{
    if (n < 0)
        return a == 1 ? 1 : (a == -1 ? ((n % 2 == 0) ? 1 : -1) : 0);
    long long r = 1;
    while (n-- > 0)
        r *= a;
    return r;
}

struct OtfVal {
    int kind;                        // 0 integer, 1 default real, 2 double
    long long i;
    float f;
    double d;
};

// one rate program (kmos_amd/otf.py opcodes) on the given counts
bool otf_eval(const int32_t *code, int ncode, const int *counts, double base, const double *userpar,
              int naux, double *out)
{
    std::vector<OtfVal> st;
    std::vector<double> aux(std::max(naux, 1), 0.0);
    int i = 0;
    while (i < ncode) {
        const int op = code[i];
        if (op == 0)
            break;
        OtfVal v{};
        switch (op) {
        case 1: v.kind = 0; v.i = code[i + 1]; st.push_back(v); i += 2; continue;
        case 2: v.kind = 1; memcpy(&v.f, &code[i + 1], 4); st.push_back(v); i += 2; continue;
        case 3: v.kind = 2; v.d = base; st.push_back(v); i += 1; continue;
        case 4: v.kind = 2; v.d = userpar[code[i + 1]]; st.push_back(v); i += 2; continue;
        case 5: v.kind = 0; v.i = counts[code[i + 1]]; st.push_back(v); i += 2; continue;
        case 6: v.kind = 2; v.d = aux[code[i + 1]]; st.push_back(v); i += 2; continue;
        case 7: if (st.empty()) return false; aux[code[i + 1]] = st.back().d; st.pop_back(); i += 2; continue;
        case 46: v.kind = 2; memcpy(&v.d, &code[i + 1], 8); st.push_back(v); i += 3; continue;
        default: break;
        }
        i += 1;
        if (st.empty())
            return false;
        OtfVal &a = st.back();
        if (op == 8) { a.f = (float)a.i; a.kind = 1; }
        else if (op == 9) { a.d = (double)a.i; a.kind = 2; }
        else if (op == 10) { a.d = (double)a.f; a.kind = 2; }
        else if (op >= 11 && op <= 13) {
            if (a.kind == 0) a.i = -a.i;
            else if (a.kind == 1) a.f = -a.f;
            else a.d = -a.d;
        } else if (op >= 20 && op <= 36) {
            if (st.size() < 2)
                return false;
            const OtfVal b = st.back();
            st.pop_back();
            OtfVal &l = st.back();
            if (op <= 31) {
                const int k = (op - 20) % 3, bop = op - k;
                if (k == 0) {
                    if (bop == 20) l.i = l.i + b.i;
                    else if (bop == 23) l.i = l.i - b.i;
                    else if (bop == 26) l.i = l.i * b.i;
                    else l.i = b.i ? l.i / b.i : 0;
                } else if (k == 1) {
                    if (bop == 20) l.f = l.f + b.f;
                    else if (bop == 23) l.f = l.f - b.f;
                    else if (bop == 26) l.f = l.f * b.f;
                    else l.f = l.f / b.f;
                } else {
                    if (bop == 20) l.d = l.d + b.d;
                    else if (bop == 23) l.d = l.d - b.d;
                    else if (bop == 26) l.d = l.d * b.d;
                    else l.d = l.d / b.d;
                }
            } else if (op == 32) l.i = otf_ipow(l.i, b.i);
            else if (op == 33) l.f = otf_powi<float>(l.f, b.i);
            else if (op == 34) l.d = otf_powi<double>(l.d, b.i);
            else if (op == 35) l.f = powf(l.f, b.f);
            else l.d = pow(l.d, b.d);
        } else if (op >= 40 && op <= 45) {
            const int dbl = (op - 40) % 2, fn = (op - 40) / 2;
            if (dbl) a.d = fn == 0 ? exp(a.d) : (fn == 1 ? log(a.d) : sqrt(a.d));
            else a.f = fn == 0 ? expf(a.f) : (fn == 1 ? logf(a.f) : sqrtf(a.f));
        } else {
            return false;
        }
    }
    if (st.empty() || st.back().kind != 2)
        return false;
    *out = st.back().d;
    return true;
}

// packed words of the device program (see the layout above)
int otf_site_word(int dx, int dy, int dz, int n1)
{
    return (dx & 0xFF) | (dy & 0xFF) << 8 | (dz & 0xFF) << 16 | (n1 - 1) << 24;
}

int otf_op_word(int kind, int dx, int dy, int dz, int ncond)
{
    return kind | (dx & 0xFF) << 2 | (dy & 0xFF) << 10 | (dz & 0xFF) << 18 | ncond << 26;
}

int otf_cond_word(int dx, int dy, int dz, int n1, int sp)
{
    return (dx & 0x7F) | (dy & 0x7F) << 7 | (dz & 0x7F) << 14 | (n1 - 1) << 21 | sp << 26;
}

// The words of otf_fast_kernel.  Leaves m->fast empty for models it does not
// take: more than 128 operations of one process or 31 on one list, more than
// four deletes on one list, an update behind an add.
void otf_build_fast(kmcg_otf_model *m, const std::vector<std::vector<std::vector<int>>> &own,
                    const std::vector<std::vector<int>> &writes)
{
    const int P = m->P;
    std::vector<int> w;
    const std::vector<int> &g = m->prog;
    m->off_fw = 0;
    w.resize(P);
    m->off_fb = (int)w.size();
    w.resize(w.size() + P);
    m->off_ft = (int)w.size();
    w.insert(w.end(), g.begin() + m->off_tbase, g.begin() + m->off_tbase + P);
    for (int p = 0; p < P; ++p) {
        w[m->off_fw + p] = (int)w.size() | (int)(writes[p].size() / 2) << 16;
        w.insert(w.end(), writes[p].begin(), writes[p].end());
    }
    for (int q = 0; q < P; ++q) {
        const int bt = g[m->off_byst + q], nb = bt >> 16;
        w[m->off_fb + q] = (int)w.size() | nb << 16;
        w.insert(w.end(), g.begin() + (bt & 0xFFFF), g.begin() + (bt & 0xFFFF) + nb * (1 + m->S));
    }
    std::map<std::vector<int>, int> pool;                // condition lists already placed
    std::vector<int> rec((size_t)P * OTF_FREC, 0);
    int reach[3] = {0, 0, 0};
    for (int p = 0; p < P; ++p) {
        int *r = &rec[(size_t)p * OTF_FREC];
        for (int j = 0; j < OTF_OPS; ++j)
            r[64 + 2 * j] = 1;
        int at = 0;
        for (int q = 0; q < P; ++q) {
            const std::vector<int> &ops = own[p][q];
            const int first = at;
            int nd = 0, nu = 0, na = 0;
            std::vector<int> gone, seen;                 // cells deleted, updated
            for (size_t i = 0; i < ops.size();) {
                const int op = ops[i], kind = op & 3, ncond = (op >> 26) & 0x3F, cellw = (op >> 2) & 0xFFFFFF;
                const std::vector<int> conds(ops.begin() + i + 1, ops.begin() + i + 1 + (kind == 3 ? ncond : 0));
                i += 1 + conds.size();
                for (int d = 0; d < 3; ++d)
                    reach[d] = std::max(reach[d], std::abs((int)(signed char)((cellw >> (8 * d)) & 0xFF)));
                const bool was = std::find(gone.begin(), gone.end(), cellw) != gone.end();
                int dup = 0, cat = 0;
                if (kind == 0) {
                    if (nu || na)
                        return;
                    if (was)
                        continue;                        // finds nothing the second time
                    gone.push_back(cellw);
                    nd += 1;
                } else if (kind == 2) {
                    if (na)
                        return;
                    if (was)
                        continue;                        // its entry is deleted in this step
                    dup = std::find(seen.begin(), seen.end(), cellw) != seen.end() ? 1 : 0;
                    seen.push_back(cellw);
                    nu += 1;
                } else {
                    na += 1;
                    const auto it = pool.emplace(conds, (int)w.size());
                    if (it.second)
                        w.insert(w.end(), conds.begin(), conds.end());
                    cat = it.first->second;
                }
                if (at >= OTF_OPS || cat > 65535)
                    return;
                r[64 + 2 * at] = kind | q << 2 | dup << 8 | (kind == 3 ? ncond : 0) << 9 | (int)((unsigned)cat << 16);
                r[64 + 2 * at + 1] = cellw;
                at += 1;
            }
            if (nd > 4 || nd + nu + na > 31)
                return;
            r[q] = first | (nd + nu + na) << 8 | nd << 16 | nu << 24;
        }
    }
    if (w.size() > 65535)
        return;
    while (w.size() % 4)
        w.push_back(0);
    m->FW = (int)w.size();
    w.insert(w.end(), rec.begin(), rec.end());
    m->fast.swap(w);
    for (int d = 0; d < 3; ++d)
        m->op_reach[d] = reach[d];
}

int otf_build(kmcg_otf_model *m)
{
    const std::vector<int32_t> &B = m->blob;
    const int P = m->P, S = m->S;
    if (m->spuck > 32 || S > 64)
        return fail(KMCG_EUNSUPPORTED, "otf engine: at most 32 sites per cell and 64 species");
    auto in = [&](long long off, long long n) { return off >= 0 && n >= 0 && off + n <= (long long)B.size(); };
    auto small = [](int v, int lim) { return v >= -lim && v <= lim; };
    std::vector<int> &g = m->prog;
    g.assign(B.begin() + B[8], B.begin() + B[8] + m->spuck);   // site defaults first
    // flat run_proc programs -> per (exec, owner) lists and per-exec writes
    std::vector<std::vector<std::vector<int>>> own(P, std::vector<std::vector<int>>(P));
    std::vector<std::vector<int>> ndel(P, std::vector<int>(P, 0)), nrest(P, std::vector<int>(P, 0));
    std::vector<std::vector<int>> writes(P);
    auto reach = [&](int dx, int dy, int dz) {
        m->reach[0] = std::max(m->reach[0], std::abs(dx));
        m->reach[1] = std::max(m->reach[1], std::abs(dy));
        m->reach[2] = std::max(m->reach[2], std::abs(dz));
    };
    // an add op and its conditions, packed; false when out of the packing's range
    auto add_op = [&](std::vector<int> &out, const int32_t *op) {
        if (op[5] > 63 || !small(op[2], 127) || !small(op[3], 127) || !small(op[4], 127))
            return false;
        out.push_back(otf_op_word(3, op[2], op[3], op[4], op[5]));
        for (int j = 0; j < op[5]; ++j) {
            const int32_t *c = op + 6 + 5 * j;
            if (c[3] < 1 || c[3] > m->spuck || c[4] < 0 || c[4] >= S || !small(c[0], 63) ||
                !small(c[1], 63) || !small(c[2], 63))
                return false;
            reach(c[0], c[1], c[2]);
            out.push_back(otf_cond_word(c[0], c[1], c[2], c[3], c[4]));
        }
        return true;
    };
    auto parse = [&](long long off, int nops, auto &&emit) -> bool {
        long long k = off;
        for (int i = 0; i < nops; ++i) {
            if (!in(k, 1))
                return false;
            const int kind = B[k];
            const int len = kind == 1 ? 7 : (kind == 3 ? (in(k, 6) ? 6 + 5 * B[k + 5] : -1) : 5);
            if (len < 0 || !in(k, len) || kind < 0 || kind > 3)
                return false;
            if (!emit(&B[k]))
                return false;
            k += len;
        }
        return true;
    };
    for (int p = 0; p < P; ++p) {
        const long long off = B[9] + 2 * p;
        if (!in(off, 2))
            return fail(KMCG_EINVAL, "otf program table out of range");
        bool after_write = false;
        const bool ok = parse(B[off + 1], B[off], [&](const int32_t *op) {
            const int kind = op[0];
            if (kind == 1) {
                if (op[5] < 0 || op[5] >= S || op[6] < 0 || op[6] >= S || op[4] < 1 || op[4] > m->spuck ||
                    !small(op[1], 127) || !small(op[2], 127) || !small(op[3], 127))
                    return false;
                writes[p].push_back(otf_site_word(op[1], op[2], op[3], op[4]));
                writes[p].push_back(op[5] | op[6] << 16);
                reach(op[1], op[2], op[3]);
                after_write = true;
                return true;
            }
            const int q = op[1];
            if (q < 0 || q >= P || !small(op[2], 127) || !small(op[3], 127) || !small(op[4], 127))
                return false;
            reach(op[2], op[3], op[4]);
            if (kind == 0) {
                if (after_write || nrest[p][q] > 0)
                    return false;                    // deletes come first
                own[p][q].push_back(otf_op_word(0, op[2], op[3], op[4], 0));
                ndel[p][q] += 1;
            } else if (kind == 2) {
                own[p][q].push_back(otf_op_word(2, op[2], op[3], op[4], 0));
                nrest[p][q] += 1;
            } else {
                if (!add_op(own[p][q], op))
                    return false;
                nrest[p][q] += 1;
            }
            return true;
        });
        if (!ok)
            return fail(KMCG_EINVAL, "bad otf program of process " + std::to_string(p + 1));
        if (writes[p].size() / 2 > 64)
            return fail(KMCG_EUNSUPPORTED, "more than 64 lattice writes in one process");
    }
    // touchup: per process its adds
    std::vector<std::vector<int>> touch(P);
    std::vector<int> ntouch(P, 0);
    const bool tok = parse(B[12], B[18], [&](const int32_t *op) {
        if (op[0] != 3 || op[1] < 0 || op[1] >= P)
            return false;
        ntouch[op[1]] += 1;
        return add_op(touch[op[1]], op);
    });
    if (!tok)
        return fail(KMCG_EINVAL, "bad otf touchup program");
    m->off_owner = (int)g.size();
    g.resize(g.size() + P * P);
    m->off_writes = (int)g.size();
    g.resize(g.size() + P);
    m->off_byst = (int)g.size();
    g.resize(g.size() + P);
    m->off_tbase = (int)g.size();
    g.resize(g.size() + P);
    m->off_touch = (int)g.size();
    g.resize(g.size() + P);
    for (int p = 0; p < P; ++p)
        for (int q = 0; q < P; ++q) {
            if (ndel[p][q] > 255 || nrest[p][q] > 255)
                return fail(KMCG_EUNSUPPORTED, "more than 255 ops of one process in one routine");
            g[m->off_owner + p * P + q] = (int)g.size() | ndel[p][q] << 16 | nrest[p][q] << 24;
            g.insert(g.end(), own[p][q].begin(), own[p][q].end());
        }
    for (int p = 0; p < P; ++p) {
        g[m->off_writes + p] = (int)g.size() | (int)(writes[p].size() / 2) << 16;
        g.insert(g.end(), writes[p].begin(), writes[p].end());
    }
    long long T = 0;
    for (int q = 0; q < P; ++q) {
        const long long rec = B[11] + 9 * q;
        if (!in(rec, 9) || !in(B[rec + 3], (long long)B[rec + 2] * (4 + S)) || !in(B[rec + 5], B[rec + 4]) ||
            !in(B[rec + 8], B[rec + 7]) || B[rec + 0] < 1 || B[rec + 1] != T)
            return fail(KMCG_EINVAL, "bad otf rate table of process " + std::to_string(q + 1));
        long long size = 1;
        for (int v = 0; v < B[rec + 7]; ++v)
            size *= (long long)B[B[rec + 8] + v] + 1;
        if (size != B[rec + 0])
            return fail(KMCG_EINVAL, "otf rate table size does not match its counts");
        g[m->off_byst + q] = (int)g.size() | B[rec + 2] << 16;
        long long reach_idx = 0;
        for (int k = 0; k < B[rec + 2]; ++k) {
            const int32_t *b = &B[B[rec + 3] + k * (4 + S)];
            if (b[3] < 1 || b[3] > m->spuck || !small(b[0], 127) || !small(b[1], 127) || !small(b[2], 127))
                return fail(KMCG_EINVAL, "bad bystander site");
            reach(b[0], b[1], b[2]);
            g.push_back(otf_site_word(b[0], b[1], b[2], b[3]));
            int most = 0;
            for (int s2 = 0; s2 < S; ++s2) {
                if (b[4 + s2] < 0)
                    return fail(KMCG_EINVAL, "negative bystander stride");
                most = std::max(most, (int)b[4 + s2]);
                g.push_back(b[4 + s2]);
            }
            reach_idx += most;
        }
        if (reach_idx >= size)
            return fail(KMCG_EINVAL, "bystander strides reach beyond the rate table of process " +
                                     std::to_string(q + 1));
        g[m->off_tbase + q] = (int)T;
        T += B[rec + 0];
    }
    for (int q = 0; q < P; ++q) {
        g[m->off_touch + q] = (int)g.size() | ntouch[q] << 16;
        g.insert(g.end(), touch[q].begin(), touch[q].end());
    }
    if (T > (1LL << 24))
        return fail(KMCG_EUNSUPPORTED, "otf rate tables too large");
    if (g.size() >= 65536 || (long long)g.size() * 4 > OTF_LDS / 2)
        return fail(KMCG_EUNSUPPORTED, "otf program too large for the engine (" + std::to_string(g.size()) +
                                       " words)");
    m->T = (int)T;
    otf_build_fast(m, own, writes);
    return KMCG_OK;
}

OtfParams otf_params(kmcg_otf_batch *b, long long steps, int mode)
{
    OtfParams p{};
    const kmcg_otf_model *m = b->m;
    p.P = m->P; p.S = m->S; p.spuck = m->spuck; p.T = m->T; p.W = (int)m->prog.size();
    p.prog = b->d_prog;
    p.off_owner = m->off_owner; p.off_writes = m->off_writes; p.off_byst = m->off_byst;
    p.off_tbase = m->off_tbase; p.off_touch = m->off_touch;
    p.fast = b->d_prog + ((m->prog.size() + 3) & ~(size_t)3);
    p.FW = m->FW; p.off_fw = m->off_fw; p.off_fb = m->off_fb; p.off_ft = m->off_ft;
    p.dims = b->d_dims; p.lat_off = b->d_lat_off; p.list_off = b->d_list_off;
    p.lat = b->d_lat; p.sites = b->d_sites; p.back = b->d_back; p.rm = b->d_rm; p.pre = b->d_pre;
    p.nsites = b->d_nsites; p.procstat = b->d_procstat; p.integ = b->d_integ; p.accum = b->d_accum;
    p.runsum = b->d_runsum; p.table = b->d_table; p.kmc_time = b->d_time; p.kmc_time_step = b->d_dt;
    p.kmc_step = b->d_step;
    p.ctr = b->d_ctr; p.seed = b->d_seed; p.stream = b->d_stream; p.status = b->d_status;
    p.rep_ids = b->d_rep; p.steps = steps; p.mode = mode; p.out = b->h_out;
    return p;
}

int otf_sync(kmcg_otf_batch *b)
{
    HIPCHK(hipSetDevice(b->device));
    HIPCHK(hipStreamSynchronize(b->stream));
    if (b->timed) {
        HIPCHK(hipEventElapsedTime(&b->last_ms, b->ev0, b->ev1));
        b->timed = false;
    }
    return KMCG_OK;
}

int otf_range(const kmcg_otf_batch *b, int32_t r0, int32_t n)
{
    if (!b || r0 < 0 || n < 1 || (long long)r0 + n > b->n)
        return fail(KMCG_EINVAL, "replica range out of the batch");
    return KMCG_OK;
}

int otf_launch(kmcg_otf_batch *b, int32_t r0, int32_t n, long long steps, int mode, bool timed)
{
    HIPCHK(hipSetDevice(b->device));
    int rc = otf_sync(b);
    if (rc)
        return rc;
    OtfParams p = otf_params(b, steps, mode);
    p.rep_ids = b->d_rep + r0;               // 0, 1, 2, ... since the batch was created
    // the steps kernel stages the program (and, when it fits, the rate
    // table) in LDS ahead of the lattice
    const size_t prog_bytes = (size_t)((p.W + 1) & ~1) * 4;
    const size_t tab_bytes = (size_t)b->m->T * 8;
    p.tab_lds = prog_bytes + tab_bytes + (size_t)b->maxV <= (size_t)OTF_LDS;
    // one lane per operation: 41 -> 24 us per step on 2048 replicas of the
    // intZGB model at 64x64 (RuO2, one 20x20 replica: 7.7 -> 5.2), and
    // faster at every size measured.  It needs the table in LDS and extents
    // on which no two offsets of the operations meet.
    const size_t fast_bytes = (size_t)((b->m->FW + 1) & ~1) * 4 + tab_bytes + OTF_OPS * 24 + (size_t)b->maxV;
    bool fast = mode < 0 && !b->m->fast.empty() && fast_bytes <= (size_t)OTF_LDS;
    for (int i = 0; i < n && fast; ++i)
        for (int d = 0; d < 3; ++d)
            fast = fast && b->dims[4 * (r0 + i) + d] >= 2 * b->m->op_reach[d] + 1;
    if (mode < 0)
        b->last_form = fast;
    if (timed)
        HIPCHK(hipEventRecord(b->ev0, b->stream));
    if (fast)
        hipLaunchKernelGGL(otf_fast_kernel, dim3(n), dim3(64), fast_bytes, b->stream, p);
    else if (mode < 0 && p.tab_lds)
        hipLaunchKernelGGL(otf_steps_kernel<true>, dim3(n), dim3(64), prog_bytes + tab_bytes + b->maxV,
                           b->stream, p);
    else if (mode < 0)
        hipLaunchKernelGGL(otf_steps_kernel<false>, dim3(n), dim3(64), prog_bytes + b->maxV, b->stream, p);
    else
        hipLaunchKernelGGL(otf_setup_kernel, dim3(n), dim3(64), (size_t)b->maxV, b->stream, p);
    HIPCHK(hipGetLastError());
    if (timed) {
        HIPCHK(hipEventRecord(b->ev1, b->stream));
        b->timed = true;
    }
    return KMCG_OK;
}

// the host evaluates each replica's tables (one per process, every count
// combination) and sends them to the device
int otf_tables(kmcg_otf_batch *b, int32_t r0, int32_t n)
{
    const kmcg_otf_model *m = b->m;
    const std::vector<int32_t> &B = m->blob;
    std::vector<double> tab((size_t)n * m->T);
    std::vector<int> counts(64);
    for (int i = 0; i < n; ++i) {
        const int r = r0 + i;
        for (int q = 0; q < m->P; ++q) {
            const long long rec = B[11] + 9 * q;
            const int size = B[rec], tbase = B[rec + 1], nused = B[rec + 7];
            if (nused > 64)
                return fail(KMCG_EUNSUPPORTED, "more than 64 bystander counts in one rate");
            for (int t = 0; t < size; ++t) {
                int rem = t;
                for (int v = 0; v < nused; ++v) {
                    counts[v] = rem % (B[B[rec + 8] + v] + 1);
                    rem /= B[B[rec + 8] + v] + 1;
                }
                double val;
                if (!otf_eval(&B[B[rec + 5]], B[rec + 4], counts.data(), b->rates[(size_t)r * m->P + q],
                              b->userpar.data() + (size_t)r * m->K, B[rec + 6], &val))
                    return fail(KMCG_EINVAL, "bad rate program of process " + std::to_string(q + 1));
                if (!(val >= 0.0))
                    return fail(KMCG_EINVAL, "otf rate of process " + std::to_string(q + 1) +
                                             " is negative or not a number");
                tab[(size_t)i * m->T + tbase + t] = val;
            }
        }
    }
    HIPCHK(hipSetDevice(b->device));
    int rc = otf_sync(b);
    if (rc)
        return rc;
    HIPCHK(hipMemcpyAsync(b->d_table + (size_t)r0 * m->T, tab.data(), tab.size() * sizeof(double),
                          hipMemcpyHostToDevice, b->stream));
    return otf_sync(b);
}

template <class T>
int otf_copy_out(kmcg_otf_batch *b, T *dst, const T *src, size_t count)
{
    int rc = otf_sync(b);
    if (rc)
        return rc;
    HIPCHK(hipMemcpy(dst, src, count * sizeof(T), hipMemcpyDeviceToHost));
    return KMCG_OK;
}

} // namespace

extern "C" {

int kmcg_otf_model_load(const int32_t *blob, int64_t nwords, kmcg_otf_model **out)
{
    if (!blob || !out || nwords < 32 || nwords > (1LL << 28))
        return fail(KMCG_EINVAL, "bad otf model blob");
    if ((uint32_t)blob[0] != 0x4B4D4347u || blob[1] != 1 || blob[2] != 2 || blob[16] != nwords)
        return fail(KMCG_EINVAL, "not an otf model blob (magic, version, backend or size)");
    auto m = new kmcg_otf_model();
    m->blob.assign(blob, blob + nwords);
    m->P = blob[3];
    m->S = blob[4];
    m->spuck = blob[6];
    m->K = blob[10];
    if (m->P < 1 || m->P > OTF_MAX_P || m->S < 1 || m->S > 64 || m->spuck < 1 || m->K < 0 ||
        blob[5] != -1) {
        delete m;
        return fail(KMCG_EUNSUPPORTED, "otf engine: 1..64 processes, one layer");
    }
    const int rc = otf_build(m);
    if (rc) {
        delete m;
        return rc;
    }
    *out = m;
    return KMCG_OK;
}

void kmcg_otf_model_free(kmcg_otf_model *m) { delete m; }

void kmcg_otf_batch_free(kmcg_otf_batch *b)
{
    if (!b)
        return;
    (void)hipSetDevice(b->device);
    if (b->stream)
        (void)hipStreamSynchronize(b->stream);
    void *ptrs[] = {b->d_prog, b->d_dims, b->d_rep, b->d_lat_off, b->d_list_off, b->d_lat, b->d_sites,
                    b->d_back, b->d_nsites, b->d_status, b->d_rm, b->d_pre, b->d_integ, b->d_accum,
                    b->d_runsum, b->d_table, b->d_time, b->d_dt, b->d_procstat, b->d_step, b->d_ctr,
                    b->d_seed, b->d_stream};
    for (void *p : ptrs)
        if (p)
            (void)hipFree(p);
    if (b->h_out)
        (void)hipHostFree(b->h_out);
    if (b->ev0)
        (void)hipEventDestroy(b->ev0);
    if (b->ev1)
        (void)hipEventDestroy(b->ev1);
    if (b->stream)
        (void)hipStreamDestroy(b->stream);
    delete b;
}

int kmcg_otf_batch_create(const kmcg_otf_model *m, int32_t n, const int32_t *sizes, int32_t device,
                          kmcg_otf_batch **out)
{
    if (!m || n < 1 || !sizes || !out)
        return fail(KMCG_EINVAL, "bad otf batch arguments");
    int count = 0;
    if (hipGetDeviceCount(&count) != hipSuccess || count < 1)
        return fail(KMCG_EINVAL, "no GPU device visible");
    if (device < 0 || device >= count)
        return fail(KMCG_EINVAL, "device index out of range");
    auto b = new kmcg_otf_batch();
    b->m = m;
    b->n = n;
    b->device = device;
    b->dims.resize(4 * (size_t)n);
    b->lat_off.resize(n);
    b->list_off.resize(n);
    for (int r = 0; r < n; ++r) {
        const int X = sizes[3 * r], Y = sizes[3 * r + 1], Z = sizes[3 * r + 2];
        const long long room = OTF_LDS - (long long)((m->prog.size() + 1) & ~(size_t)1) * 4;
        if (X < 1 || Y < 1 || Z < 1 || X < m->reach[0] || Y < m->reach[1] || Z < m->reach[2] ||
            (long long)X * Y * Z * m->spuck > std::min<long long>(OTF_MAX_V, room)) {
            delete b;
            return fail(KMCG_EINVAL, "lattice size of replica " + std::to_string(r) +
                                     " outside the engine's range (each extent at least the model's "
                                     "largest offset; at most " + std::to_string(std::min<long long>(OTF_MAX_V, room)) +
                                     " sites beside this model's program in 64 KiB of LDS)");
        }
        const int C = X * Y * Z;
        b->dims[4 * r] = X; b->dims[4 * r + 1] = Y; b->dims[4 * r + 2] = Z; b->dims[4 * r + 3] = C;
        b->lat_off[r] = b->lat_total;
        b->lat_total += (long long)C * m->spuck;
        b->list_off[r] = b->list_total;
        b->list_total += otf_row(C) * m->P;
        b->maxV = std::max(b->maxV, C * m->spuck);
    }
    b->rates.assign((size_t)n * m->P, 0.0);
    b->userpar.assign((size_t)n * std::max(m->K, 1), 0.0);
    auto bail = [&](int code, const std::string &msg) {
        kmcg_otf_batch_free(b);
        return fail(code, msg);
    };
    if (hipSetDevice(device) != hipSuccess || hipStreamCreate(&b->stream) != hipSuccess ||
        hipEventCreate(&b->ev0) != hipSuccess || hipEventCreate(&b->ev1) != hipSuccess)
        return bail(KMCG_EHIP, "stream or event creation failed");
    const size_t P = m->P;
    std::vector<int> progs(m->prog);                     // the program, then the fast kernel's words
    progs.resize((progs.size() + 3) & ~(size_t)3, 0);
    progs.insert(progs.end(), m->fast.begin(), m->fast.end());
    struct A { void **p; size_t bytes; } allocs[] = {
        {(void **)&b->d_prog, progs.size() * sizeof(int)},
        {(void **)&b->d_dims, b->dims.size() * sizeof(int)},
        {(void **)&b->d_rep, (size_t)n * sizeof(int)},
        {(void **)&b->d_lat_off, (size_t)n * sizeof(long long)},
        {(void **)&b->d_list_off, (size_t)n * sizeof(long long)},
        {(void **)&b->d_lat, (size_t)b->lat_total},
        {(void **)&b->d_sites, (size_t)b->list_total * sizeof(int)},
        {(void **)&b->d_back, (size_t)b->list_total * sizeof(int)},
        {(void **)&b->d_rm, (size_t)b->list_total * sizeof(double)},
        {(void **)&b->d_pre, (size_t)(b->list_total / OTF_BLK) * sizeof(double)},
        {(void **)&b->d_nsites, n * P * sizeof(int)},
        {(void **)&b->d_status, (size_t)n * sizeof(int)},
        {(void **)&b->d_integ, n * P * sizeof(double)},
        {(void **)&b->d_accum, n * P * sizeof(double)},
        {(void **)&b->d_runsum, n * P * sizeof(double)},
        {(void **)&b->d_table, (size_t)n * std::max(m->T, 1) * sizeof(double)},
        {(void **)&b->d_time, (size_t)n * sizeof(double)},
        {(void **)&b->d_dt, (size_t)n * sizeof(double)},
        {(void **)&b->d_procstat, n * P * sizeof(long long)},
        {(void **)&b->d_step, (size_t)n * sizeof(long long)},
        {(void **)&b->d_ctr, (size_t)n * sizeof(unsigned long long)},
        {(void **)&b->d_seed, (size_t)n * sizeof(unsigned)},
        {(void **)&b->d_stream, (size_t)n * sizeof(unsigned)},
    };
    for (auto &a : allocs)
        if (hipMalloc(a.p, std::max(a.bytes, (size_t)8)) != hipSuccess)
            return bail(KMCG_ENOMEM, "device allocation failed for an otf batch");
    if (hipHostMalloc((void **)&b->h_out, (size_t)n * OTF_OUT(m->P) * sizeof(double), hipHostMallocDefault) != hipSuccess)
        return bail(KMCG_ENOMEM, "pinned host allocation failed for an otf batch");
    memset(b->h_out, 0, (size_t)n * OTF_OUT(m->P) * sizeof(double));
    for (int r = 0; r < n; ++r)
        ((long long *)b->h_out)[(size_t)(r + 1) * OTF_OUT(m->P) - 1] = -1;     // not initialised
    std::vector<int> iota(n);
    for (int r = 0; r < n; ++r)
        iota[r] = r;
    if (hipMemcpy(b->d_prog, progs.data(), progs.size() * sizeof(int), hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(b->d_dims, b->dims.data(), b->dims.size() * sizeof(int), hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(b->d_rep, iota.data(), n * sizeof(int), hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(b->d_lat_off, b->lat_off.data(), n * sizeof(long long), hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(b->d_list_off, b->list_off.data(), n * sizeof(long long), hipMemcpyHostToDevice) != hipSuccess ||
        hipMemset(b->d_nsites, 0, n * P * sizeof(int)) != hipSuccess ||
        hipMemset(b->d_rm, 0, (size_t)b->list_total * sizeof(double)) != hipSuccess ||
        hipMemset(b->d_runsum, 0, n * P * sizeof(double)) != hipSuccess ||
        hipMemset(b->d_table, 0, (size_t)n * std::max(m->T, 1) * sizeof(double)) != hipSuccess ||
        hipMemset(b->d_status, 0xff, (size_t)n * sizeof(int)) != hipSuccess)
        return bail(KMCG_EHIP, "otf batch set-up copies failed");
    *out = b;
    return KMCG_OK;
}

int kmcg_otf_init(kmcg_otf_batch *b, int32_t r0, int32_t n, const uint32_t *seeds, const uint32_t *streams)
{
    int rc = otf_range(b, r0, n);
    if (rc)
        return rc;
    if (!seeds || !streams)
        return fail(KMCG_EINVAL, "seeds and streams are required");
    if ((rc = otf_sync(b)))
        return rc;
    HIPCHK(hipMemcpy(b->d_seed + r0, seeds, n * sizeof(unsigned), hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(b->d_stream + r0, streams, n * sizeof(unsigned), hipMemcpyHostToDevice));
    if ((rc = otf_launch(b, r0, n, 0, 0, false)))
        return rc;
    return otf_sync(b);
}

int kmcg_otf_set_params(kmcg_otf_batch *b, int32_t r0, int32_t n, const double *rates, const double *userpar)
{
    int rc = otf_range(b, r0, n);
    if (rc)
        return rc;
    const int P = b->m->P, K = b->m->K;
    if (!rates || (K > 0 && !userpar))
        return fail(KMCG_EINVAL, "rates (and parameters) are required");
    for (long long i = 0; i < (long long)n * P; ++i)
        if (!(rates[i] >= 0.0) || !std::isfinite(rates[i]))
            return fail(KMCG_EINVAL, "rate constants must be finite and non-negative");
    for (long long i = 0; i < (long long)n * K; ++i)
        if (!std::isfinite(userpar[i]))
            return fail(KMCG_EINVAL, "parameters must be finite");
    std::vector<double> old_r(b->rates), old_u(b->userpar);
    std::copy(rates, rates + (size_t)n * P, b->rates.begin() + (size_t)r0 * P);
    if (K > 0)
        std::copy(userpar, userpar + (size_t)n * K, b->userpar.begin() + (size_t)r0 * K);
    if ((rc = otf_tables(b, r0, n))) {
        b->rates.swap(old_r);
        b->userpar.swap(old_u);
        return rc;
    }
    if (b->status(r0) == -1)
        return KMCG_OK;                   // not initialised yet: init builds the lists
    if ((rc = otf_launch(b, r0, n, 0, 2, false)))
        return rc;
    return otf_sync(b);
}

int kmcg_otf_set_config(kmcg_otf_batch *b, int32_t r0, int32_t n, const int8_t *config)
{
    int rc = otf_range(b, r0, n);
    if (rc)
        return rc;
    if (!config)
        return fail(KMCG_EINVAL, "config is required");
    long long total = 0;
    for (int i = 0; i < n; ++i)
        total += (long long)b->dims[4 * (r0 + i) + 3] * b->m->spuck;
    for (long long i = 0; i < total; ++i)
        if (config[i] < 0 || config[i] >= b->m->S)
            return fail(KMCG_EINVAL, "species ids must be 0..S-1");
    if ((rc = otf_sync(b)))
        return rc;
    for (int i = 0; i < n; ++i)
        if (b->status(r0 + i) == -1)
            return fail(KMCG_EINVAL, "set_config before init");
    HIPCHK(hipMemcpy(b->d_lat + b->lat_off[r0], config, total, hipMemcpyHostToDevice));
    if ((rc = otf_launch(b, r0, n, 0, 1, false)))
        return rc;
    return otf_sync(b);
}

int kmcg_otf_run(kmcg_otf_batch *b, int32_t r0, int32_t n, int64_t steps)
{
    int rc = otf_range(b, r0, n);
    if (rc)
        return rc;
    if (steps < 0)
        return fail(KMCG_EINVAL, "steps must be non-negative");
    if ((rc = otf_sync(b)))
        return rc;
    for (int i = 0; i < n; ++i)
        if (b->status(r0 + i) == -1)
            return fail(KMCG_EINVAL, "run before init");
    return otf_launch(b, r0, n, steps, -1, true);
}

int kmcg_otf_sync(kmcg_otf_batch *b)
{
    if (!b)
        return fail(KMCG_EINVAL, "null batch");
    return otf_sync(b);
}

int kmcg_otf_last_form(const kmcg_otf_batch *b, int32_t *form)
{
    if (!b || !form)
        return fail(KMCG_EINVAL, "null argument");
    *form = b->last_form;
    return KMCG_OK;
}

int kmcg_otf_last_run_ms(kmcg_otf_batch *b, float *ms)
{
    if (!b || !ms)
        return fail(KMCG_EINVAL, "bad arguments");
    int rc = otf_sync(b);
    *ms = b->last_ms;
    return rc;
}

int kmcg_otf_get_scalars(kmcg_otf_batch *b, int32_t r, double *kmc_time, double *kmc_time_step, int64_t *kmc_step,
                         int32_t *status)
{
    int rc = otf_range(b, r, 1);
    if (rc)
        return rc;
    // (the read-back words are written by the kernels that change them: a
    // getter costs no copy of its own, 15 us each)
    if ((rc = otf_sync(b)))
        return rc;
    const long long *o = b->out(r) + 4 * b->m->P;
    memcpy(kmc_time, o, 8);
    memcpy(kmc_time_step, o + 1, 8);
    *kmc_step = o[2];
    *status = (int32_t)o[3];
    return KMCG_OK;
}

int kmcg_otf_get_lattice(kmcg_otf_batch *b, int32_t r, int8_t *out)
{
    int rc = otf_range(b, r, 1);
    if (rc)
        return rc;
    return otf_copy_out(b, (signed char *)out, b->d_lat + b->lat_off[r], (size_t)b->dims[4 * r + 3] * b->m->spuck);
}

int kmcg_otf_get_counters(kmcg_otf_batch *b, int32_t r, int32_t *nr_of_sites, int64_t *procstat, double *integ,
                          double *accum)
{
    int rc = otf_range(b, r, 1);
    if (rc)
        return rc;
    const size_t P = b->m->P;
    if ((rc = otf_sync(b)))
        return rc;
    const long long *o = b->out(r);
    memcpy(integ, o, P * 8);
    memcpy(accum, o + P, P * 8);
    for (size_t p = 0; p < P; ++p) {
        procstat[p] = o[2 * P + p];
        nr_of_sites[p] = (int32_t)o[3 * P + p];
    }
    return KMCG_OK;
}

int kmcg_otf_get_avail(kmcg_otf_batch *b, int32_t r, int32_t *sites, int32_t *back, double *rates_matrix)
{
    int rc = otf_range(b, r, 1);
    if (rc)
        return rc;
    const kmcg_otf_model *m = b->m;
    const int P = m->P, C = b->dims[4 * r + 3], V = C * m->spuck;
    const size_t R = (size_t)otf_row(C);
    std::vector<int> s(P * R), bk(P * R);
    std::vector<double> rm(P * R), run(P);
    if ((rc = otf_copy_out(b, s.data(), b->d_sites + b->list_off[r], s.size())) ||
        (rc = otf_copy_out(b, bk.data(), b->d_back + b->list_off[r], bk.size())) ||
        (rc = otf_copy_out(b, rm.data(), b->d_rm + b->list_off[r], rm.size())) ||
        (rc = otf_copy_out(b, run.data(), b->d_runsum + (size_t)r * P, (size_t)P)))
        return rc;
    // avail_sites(p, i, 1): site numbers (site 1 of the cell), avail_sites(p,
    // site, 2): list positions; rates_matrix(p, 1:V) and (p, V+1)
    for (int p = 0; p < P; ++p) {
        for (int i = 0; i < V; ++i) {
            sites[(size_t)p * V + i] = 0;
            back[(size_t)p * V + i] = 0;
            rates_matrix[(size_t)p * (V + 1) + i] = 0.0;
        }
        for (int i = 0; i < C; ++i) {
            const int cell1 = s[p * R + i];
            sites[(size_t)p * V + i] = cell1 ? (cell1 - 1) * m->spuck + 1 : 0;
            back[(size_t)p * V + (size_t)i * m->spuck] = bk[p * R + i];
            rates_matrix[(size_t)p * (V + 1) + i] = rm[p * R + i];
        }
        rates_matrix[(size_t)p * (V + 1) + V] = run[p];
    }
    return KMCG_OK;
}

int kmcg_otf_get_table(kmcg_otf_batch *b, int32_t r, double *out)
{
    int rc = otf_range(b, r, 1);
    if (rc)
        return rc;
    return otf_copy_out(b, out, b->d_table + (size_t)r * b->m->T, (size_t)b->m->T);
}

int kmcg_otf_model_info(const kmcg_otf_model *m, int32_t *info4)
{
    if (!m || !info4)
        return fail(KMCG_EINVAL, "bad arguments");
    info4[0] = m->P;
    info4[1] = m->S;
    info4[2] = m->K;
    info4[3] = m->T;
    return KMCG_OK;
}

} // extern "C"
