// group.hip -- BiCGStab of systems that fit on the chip, one launch per
// solve: every segment is iterated by a group of work-groups that stay
// resident until it stops.
//
// What bounds the launched iteration (krylov.hip) on such systems is not
// memory: six to eight dependent launches of a few microseconds each, and a
// host read of the flags per batch, 37-48 us per iteration whatever the size
// below about 200,000 unknowns.  Here a lane owns a face.  Its matrix rows,
// its p and r, and copies of its neighbours' p and r live in registers (x and
// r* in LDS); an iteration is the merged recurrence (FIN_*_MERGED) with two
// exchanges.  In each the lanes publish one vector (Ap, then As), the
// work-groups publish their partial dot products, and every work-group reads
// all partial sums and the published values of its neighbours; each lane then
// updates the copies of its neighbours' vectors with the arithmetic of their
// owners, so p and s are never exchanged themselves.
//
// * Published values are their own flags (device.hpp): no fence, no counter,
//   and the gather of the neighbours overlaps the reduction.  There are
//   GROUP_ROT copies; one is cleared by its owner once every work-group has
//   posted the epoch after it, three epochs before it is used again.
// * All work-groups add the partial sums in one order, so all take the same
//   decisions and leave the loop together.
// * Faces are taken along a space-filling curve (group_order): most
//   neighbours are in the same work-group and come through LDS.
// * Work-groups take their share by ticket, the segments' shares in a row,
//   largest segment first, and the next one when theirs is done: the earliest
//   unfinished segment has all its shares taken once earlier ones are done,
//   so a batch may have many more shares than work-groups fit at once.
// * Nothing else on the GPU is waited for: when another launch holds places
//   that a segment needs and neither gets on, no iteration of this launch
//   happens for 5 ms and the waits give up.  The segment is marked, every
//   work-group leaves, and the host restarts it with the launched iteration
//   from the iterate it has (and keeps to that for some solves where the
//   next try gives up too).
//
// Measured (MI355X, whole trajectories as in perf/cases.py, ms, and us per
// iteration, by launches -> in one launch): 64 x 64 x 2 triangles, 3 steps 1.82 ->
// 0.48 (31 -> 8.1); 201 x 201 x 2, 2 steps 3.94 -> 0.84 (26 -> 6.4); 21^3 x 6
// tetrahedra n = 1, 2 steps 9.8 -> 1.87 (27 -> 5.2); 20^3 x 6 n = 2, FP32, 6 steps
// 32.9 -> 7.7 (34 -> 8.0); 20^3 voxels n = 3, 3.53 -> 1.20 (32 -> 11); 32 ragged 2-D
// instances 36.4 -> 14.2.  An exchange takes 2.4 us with 200 work-groups: 0.5 us
// of arithmetic, 0.4 us of work-group sums, the rest from the post of the
// slowest work-group to its sum in every other one.  Tried: neighbours polled
// only after the sums are in (10 us per iteration where 8 were needed then);
// faces in the mesh order (gathers 2.3 us instead of 1.6).
#include <algorithm>
#include <type_traits>

#include "common.hpp"
#include "device.hpp"

namespace mhfem {

constexpr int GROUP_ROT = 4;  // rotating copies of the published vectors and partial sums
constexpr int GROUP_REP = 8;  // copies of the partial sums, each read by every 8th work-group
// Pause before the first look at the others' values, in 64 cycles (0.53 us at
// 2.4 GHz).  They cannot be there sooner than a store and a load take, and
// looks before that only load the fabric that carries them: ms per pass with
// 0 / 12 / 16 / 18 / 19 / 20 / 21 / 22 / 24: 114,000 faces of tetrahedra, 357
// iterations 2.79 / 2.28 / 1.92 / 1.87 / 1.85 / 1.87 / 1.90 / 1.92 / 1.95; 121,600
// of triangles, 131 iterations 1.35 / 1.11 / 1.01 / 0.95 / 0.87 / 0.85 / 0.84 /
// 0.83 / 0.83; FP32, 98,400 faces n = 2, 958 iterations 10.0 / 8.66 / 7.92 / 7.68 /
// 7.58 / 7.67 / 7.74 / 7.77 / 7.82; 32 ragged instances 18.6 / 15.7 / 14.4 / 14.0 /
// 14.1 / 14.3 / 14.4 / 14.6 / 14.8.  Later looks gain nothing from longer pauses
// (4 or 8 instead of 1: 2-20 % slower).
constexpr int GROUP_FIRST_LOOK = 20;
constexpr int GROUP_ND = 4;   // dot products of a reduction, at most

// partial sums a wavefront adds, per dot product: BS / 256 wavefronts for each
// of GROUP_ND dots cover the largest group (one work-group per CU of 256)
constexpr int group_slots(int bs) { return bs <= 256 ? 256 : 128; }
// Threads of a part: a work-group of 1024 takes two parts of a segment, whose
// sums it posts separately, so that the order of a segment's sums does not
// depend on the threads its batch is run with.
constexpr int part_threads(int bs) { return std::min(bs, 512); }

// Where a lane's matrix rows stay between products: in registers; in LDS, with
// at most LDS_FACES faces per work-group; or in memory (the L2), read in each
// product.
enum { HOLD_MEMORY = 0, HOLD_REGS = 1, HOLD_LDS = 2 };
constexpr int LDS_FACES = 128;

struct GroupView {
    int total;               // shares, one per ticket
    int64_t rows;
    const GroupTask *task;   // per ticket
    const int *face, *pos;   // the face at a position of the groups' order, and its inverse
    const int2 *seg;         // per segment: first slot (of GROUP_ROT * GROUP_ND * parts), parts
    int *ticket;             // [0]
    unsigned *beat;          // [0]: iterations of every segment of the launch
    double *slots;
    double *sc;
    unsigned long long wait_ticks;  // bound of a wait, 0: every wait gives up at its first pause
};

// Values of one face moved through memory as 8- or 4-byte words with
// device-coherent accesses; a component that still holds the sentinel has not
// been written yet.
template <typename T, int N>
struct FaceWords {
    using U = std::conditional_t<(sizeof(T) * N) % 8 == 0, unsigned long long, unsigned int>;
    static constexpr int M = (int)(sizeof(T) * N / sizeof(U));
    union {
        U w[M];
        T v[N];
    };
    __device__ FaceWords() {}
};
template <typename T, int N>
__device__ __forceinline__ void publish(T *dst, const Pack<T, N> &a)
{
    FaceWords<T, N> f;
#pragma unroll
    for (int i = 0; i < N; i++) f.v[i] = is_sentinel(a.v[i]) ? (T)__builtin_nan("") : a.v[i];
    auto *q = reinterpret_cast<typename FaceWords<T, N>::U *>(dst);
#pragma unroll
    for (int m = 0; m < FaceWords<T, N>::M; m++) coherent_store(q + m, f.w[m]);
}
template <typename T, int N>
__device__ __forceinline__ Pack<T, N> look(const T *src)
{
    FaceWords<T, N> f;
    auto *q = reinterpret_cast<const typename FaceWords<T, N>::U *>(src);
#pragma unroll
    for (int m = 0; m < FaceWords<T, N>::M; m++) f.w[m] = coherent_load(q + m);
    Pack<T, N> a;
#pragma unroll
    for (int i = 0; i < N; i++) a.v[i] = f.v[i];
    return a;
}
template <typename T, int N>
__device__ __forceinline__ void unpublish(T *dst)
{
    FaceWords<T, N> f;
#pragma unroll
    for (int i = 0; i < N; i++) f.v[i] = sentinel_value<T>();
    auto *q = reinterpret_cast<typename FaceWords<T, N>::U *>(dst);
#pragma unroll
    for (int m = 0; m < FaceWords<T, N>::M; m++) coherent_store(q + m, f.w[m]);
}

// a value every lane of the wavefront holds, moved to scalar registers
__device__ __forceinline__ double uniform(double v)
{
    const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
    const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)b), hi = __builtin_amdgcn_readfirstlane((unsigned)(b >> 32));
    return __builtin_bit_cast(double, (unsigned long long)hi << 32 | lo);
}

// every memory access issued so far is complete (the builtin, so that the
// compiler's own count of outstanding accesses starts at zero here)
__device__ __forceinline__ void memory_done()
{
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
    asm volatile("" ::: "memory");
}

// bounded waiting: gives up once nothing in the launch has iterated for
// g.wait_ticks, or a work-group of the segment has given up
struct GroupWait {
    const GroupView &g;
    double *fail;  // the segment's S_FAIL
    unsigned long long t0 = 0;
    unsigned beat = 0;
    int idle = 0;
    bool gave_up = false;
    __device__ GroupWait(const GroupView &v, double *f) : g(v), fail(f) {}
    __device__ __forceinline__ bool pause()
    {
        __builtin_amdgcn_s_sleep(1);
        if ((++idle & 63) == 0 || g.wait_ticks == 0) {
            const unsigned long long now = __builtin_amdgcn_s_memrealtime();
            const unsigned b = coherent_load(g.beat);
            if (t0 == 0 || b != beat) {
                t0 = now;
                beat = b;
            } else if (now - t0 > g.wait_ticks) {
                gave_up = true;
            }
            if (g.wait_ticks == 0) gave_up = true;
            if (coherent_load(fail) != 0.0) gave_up = true;
            if (gave_up) coherent_store(fail, 1.0);
        }
        return gave_up;
    }
};

// The arithmetic of an iteration is written out, so that every instantiation
// (threads, where the rows are held, batch or not) gives the same bits: a
// batch may run its instances in another one than their own contexts do.
#pragma clang fp contract(off)
__device__ __forceinline__ double fmadd(double a, double b, double c) { return __builtin_fma(a, b, c); }
__device__ __forceinline__ float fmadd(float a, float b, float c) { return __builtin_fmaf(a, b, c); }

// One share of a segment, from the next ticket; false: no share is left, or a
// wait gave up.
template <typename T, int N, int W, int BS, int HOLD, bool BATCH>
__device__ __forceinline__ bool bicg_share(const SellView<T> &A, const GroupView &g, T *__restrict__ xg,
                                           T *__restrict__ rg, T *__restrict__ pg, const T *__restrict__ r_ast,
                                           const T *__restrict__ qg, T *pub)
{
    constexpr int NW = BS / 64, SLOTS = group_slots(BS), PT = part_threads(BS), NP = BS / PT;
    __shared__ int s_ticket, s_fail;
    __shared__ double part[2][GROUP_ND][NW], tot[2][GROUP_ND][NW / GROUP_ND];
    __shared__ Pack<T, N> mine[2][BS + 1];  // the work-group's own published values; zeros in the last
    __shared__ Pack<T, N> own[2][BS];   // x and r* of each lane
    // HOLD_LDS: the matrix rows, entry by entry across the lanes with a face
    __shared__ T rows[HOLD == HOLD_LDS ? W * N * N * LDS_FACES : 1];
    const int tid = threadIdx.x, lane = tid & 63, wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    if constexpr (BATCH) __syncthreads();  // the last share's sums have been read
    if (tid == 0) {
        s_ticket = atomicAdd(g.ticket, 1);
        s_fail = 0;
    }
    if (tid < 2)
#pragma unroll
        for (int i = 0; i < N; i++) mine[tid][BS].v[i] = T(0);
    if (tid < 2 * GROUP_ND * (NW / GROUP_ND)) (&tot[0][0][0])[tid] = 0.0;  // chunks past the group stay zero
    __syncthreads();
    const int ticket = __builtin_amdgcn_readfirstlane(s_ticket);
    if (ticket >= g.total) return false;
    const GroupTask task = g.task[ticket];
    double *sc = g.sc + (int64_t)task.seg * NSLOTS;
    if (halted(sc)) return true;
    const int G = g.seg[task.seg].y;
    double *slots = g.slots + g.seg[task.seg].x;
    const int at = task.p0 + tid / PT * task.part + tid % PT;  // position in the groups' order
    const bool valid = at < task.p1 && (NP == 1 || tid % PT < task.part);
    const int parts = NP > 1 && task.p0 + task.part < task.p1 ? NP : 1;
    const int f = valid ? g.face[at] : 0;

    // ---- the face's matrix rows and its state; neighbours' p and r
    int col[W];  // the neighbour's row in the published vector, or -1 - its lane when this work-group has it
    Pack<T, N * N> val[HOLD == HOLD_REGS ? W : 1];
    Pack<T, (N > 1 ? N * (N - 1) : 1)> dg;
    Pack<T, N> p, r, pn[W], rn[W];
    int w = 0;
#pragma unroll
    for (int i = 0; i < N; i++) p.v[i] = r.v[i] = T(0);
    if constexpr (N > 1) {
#pragma unroll
        for (int i = 0; i < N * (N - 1); i++) dg.v[i] = T(0);
    }
    int64_t base = 0;
    if (valid) {
        base = A.slice_ptr[f >> 6] + (f & 63);
        w = A.slice_width[f >> 6];
    }
    // the direction after a reliable update: r + S_BFIX q
    const T fix = qg ? (T)uniform(sc[S_BFIX]) : T(0);
    auto direction = [&](int face, const Pack<T, N> &res) {
        Pack<T, N> d = ld<T, N>((qg ? qg : pg) + (int64_t)face * N);
        if (qg) {
#pragma unroll
            for (int i = 0; i < N; i++) d.v[i] = fmadd(fix, d.v[i], res.v[i]);
        }
        return d;
    };
    unsigned remote = 0;  // neighbours in other work-groups
    bool alone = true;    // no neighbour but itself (padding)
#pragma unroll
    for (int k = 0; k < W; k++) {
        col[k] = k < w ? A.col[base + (int64_t)k * 64] : f;
        if constexpr (HOLD == HOLD_REGS) {
#pragma unroll
            for (int i = 0; i < N * N; i++) val[k].v[i] = T(0);
        }
#pragma unroll
        for (int i = 0; i < N; i++) pn[k].v[i] = rn[k].v[i] = T(0);
        if (k < w) {
            if constexpr (HOLD == HOLD_REGS) val[k] = ld<T, N * N>(A.val + (base + (int64_t)k * 64) * (N * N));
            if constexpr (HOLD == HOLD_LDS) {
                const Pack<T, N * N> row = ld<T, N * N>(A.val + (base + (int64_t)k * 64) * (N * N));
#pragma unroll
                for (int i = 0; i < N * N; i++) rows[(k * N * N + i) * LDS_FACES + tid] = row.v[i];
            }
            rn[k] = ld<T, N>(rg + (int64_t)col[k] * N);
            pn[k] = direction(col[k], rn[k]);
        }
        alone = alone && col[k] == f;
        // Slots past the face's width read zeros: the product multiplies
        // them by stored zeros, and any other value kept there would follow a
        // recurrence that the solution does not bound (one overflow, and
        // 0 Inf = NaN).
        col[k] = k < w ? g.pos[col[k]] : -1 - BS;
        if (col[k] < 0) continue;
        if (col[k] < task.p0 || col[k] >= task.p1) remote |= 1u << k;
        else {
            const int d = col[k] - task.p0;
            col[k] = -1 - (NP > 1 && d >= task.part ? d - task.part + PT : d);
        }
    }
    // The pattern is symmetric but for faces without neighbours (all rows
    // Dirichlet), which their neighbours read: those faces and the ones that
    // read other work-groups' faces are published.
    const bool shared_face = valid && (remote != 0 || alone);
    own[0][tid] = own[1][tid] = p;
    if (valid) {
        r = ld<T, N>(rg + (int64_t)f * N);
        p = direction(f, r);
        own[0][tid] = ld<T, N>(xg + (int64_t)f * N);
        own[1][tid] = ld<T, N>(r_ast + (int64_t)f * N);
        if constexpr (N > 1) dg = ld<T, N *(N - 1)>(A.val + A.diag_base + (int64_t)f * N * (N - 1));
    }
    double rho = uniform(sc[S_RHO]), rho_old = uniform(sc[S_RHO_OLD]), alpha = uniform(sc[S_ALPHA]),
           omega = uniform(sc[S_OMEGA]), beta = uniform(sc[S_BETA]);
    double resid = 0.0, it = uniform(sc[S_IT]), brk = uniform(sc[S_BREAK]);
    double inv_pap = 0.0;  // alpha / rho
    const double bnorm = uniform(sc[S_BNORM]), tol = uniform(sc[S_TOL]), maxit = uniform(sc[S_MAXIT]),
                 rast_sq = uniform(sc[S_RAST_SQ]);
    double done = 0.0, restart = 0.0;
    const double eps2 = 2.220446049250313e-16 * 2.220446049250313e-16;
    // every read of the arrays that the segment's work-groups write at the
    // end is complete before this work-group's first partial sums go out
    memory_done();

    auto product = [&](const Pack<T, N> &own, const Pack<T, N>(&nb)[W]) {
        Pack<T, N> y = own;
        if constexpr (N > 1) {
#pragma unroll
            for (int i = 0; i < N; i++)
#pragma unroll
                for (int j = 0; j < N; j++)
                    if (j != i) y.v[i] = fmadd(dg.v[i * (N - 1) + (j < i ? j : j - 1)], own.v[j], y.v[i]);
        }
#pragma unroll
        for (int k = 0; k < W; k++) {
            constexpr int R = HOLD == HOLD_REGS ? 1 : 0;
            if constexpr (HOLD == HOLD_MEMORY) {
                if (k < w) val[0] = ld<T, N * N>(A.val + (base + (int64_t)k * 64) * (N * N));
            }
            if constexpr (HOLD == HOLD_LDS) {
                if (k < w) {
#pragma unroll
                    for (int i = 0; i < N * N; i++) val[0].v[i] = rows[(k * N * N + i) * LDS_FACES + tid];
                }
            }
            if (HOLD == HOLD_REGS || k < w) {
#pragma unroll
                for (int i = 0; i < N; i++)
#pragma unroll
                    for (int j = 0; j < N; j++) y.v[i] = fmadd(val[R * k].v[i * N + j], nb[k].v[j], y.v[i]);
            }
        }
        return y;
    };
    GroupWait wait(g, sc + S_FAIL);
    int e = 0;  // epoch: one per reduction
    // publishes y, sums the partials of ND dots over the group into tot and
    // gathers the neighbours' published values; false: a wait gave up
    auto exchange = [&](const Pack<T, N> &y, auto &acc, auto NDC, Pack<T, N>(&nb)[W]) {
        constexpr int ND = decltype(NDC)::value;
        const int rot = e & (GROUP_ROT - 1), par = e & 1;
        T *pb = pub + (int64_t)rot * g.rows;
        if (shared_face) publish<T, N>(pb + (int64_t)at * N, y);
        mine[par][tid] = y;
        const double ws = sums_wave<ND>(acc);
        if ((lane & (64 / ND - 1)) == 0) part[par][lane / (64 / ND)][wid] = ws;
        __syncthreads();
        // (The two forms are apart for the compiler's sake: with the second for
        // both, the kernels of one part are 1-2 % slower.)
        if constexpr (NP == 1) {
            if (tid < ND * GROUP_REP) {
                double s = part[par][tid % ND][0];
#pragma unroll
                for (int q = 1; q < NW; q++) s += part[par][tid % ND][q];
                if (is_sentinel(s)) s = __builtin_nan("");
                coherent_store(slots + (((int64_t)(tid / ND) * GROUP_ROT + rot) * GROUP_ND + tid % ND) * G + task.rank,
                               s);
            }
        } else if (tid < parts * ND * GROUP_REP) {
            const int h = tid / (ND * GROUP_REP), rep = tid / ND % GROUP_REP;
            double s = part[par][tid % ND][h * (PT / 64)];
#pragma unroll
            for (int q = 1; q < PT / 64; q++) s += part[par][tid % ND][h * (PT / 64) + q];
            if (is_sentinel(s)) s = __builtin_nan("");
            coherent_store(slots + (((int64_t)rep * GROUP_ROT + rot) * GROUP_ND + tid % ND) * G + task.rank + h, s);
        }
#pragma unroll
        for (int k = 0; k < W; k++)
            nb[k] = mine[par][min((unsigned)~col[k], (unsigned)BS)];  // (zeros until a remote one is there)
        // Polls for the neighbours' values in other work-groups and, in wave
        // d + ND c, for the sums of dot d of SLOTS work-groups: each round looks
        // at everything still missing with one wait.
        unsigned pend = remote, pd = 0;
        const int dot = wid & (ND - 1), chunk = wid / ND * SLOTS;
        const double *row =
            slots + (((int64_t)(task.rank / NP % GROUP_REP) * GROUP_ROT + rot) * GROUP_ND + dot) * G + chunk;
        double v[SLOTS / 64];
#pragma unroll
        for (int q = 0; q < SLOTS / 64; q++) {
            v[q] = 0.0;
            if (chunk + q * 64 + lane < G) pd |= 1u << q;
        }
        __builtin_amdgcn_s_sleep(GROUP_FIRST_LOOK);
        for (;;) {
#pragma unroll
            for (int k = 0; k < W; k++)
                if (pend >> k & 1u) nb[k] = look<T, N>(pb + (int64_t)col[k] * N);
#pragma unroll
            for (int q = 0; q < SLOTS / 64; q++)
                if (pd >> q & 1u) v[q] = coherent_load(row + q * 64 + lane);
#pragma unroll
            for (int k = 0; k < W; k++) {
                bool there = true;
#pragma unroll
                for (int i = 0; i < N; i++) there = there && !is_sentinel(nb[k].v[i]);
                if (there) pend &= ~(1u << k);
            }
#pragma unroll
            for (int q = 0; q < SLOTS / 64; q++)
                if (!is_sentinel(v[q])) pd &= ~(1u << q);
            if (!__any((pend | pd) != 0)) break;
            if (wait.pause()) {
                if (lane == 0) s_fail = 1;
                break;
            }
        }
        wait.t0 = 0;
        if (chunk < G) {
            double one[1] = {v[0]};
#pragma unroll
            for (int q = 1; q < SLOTS / 64; q++) one[0] += v[q];
            const double s = sums_wave<1>(one);
            if (lane == 0) tot[par][dot][wid / ND] = s;
        }
        // the clearing stores of the previous epoch are complete before the
        // work-group posts its next partial sums
        memory_done();
        __syncthreads();
        // every work-group has posted this epoch, so none still reads the
        // previous one: its copies are cleared, for epoch e + 3
        const int old = (e + GROUP_ROT - 1) & (GROUP_ROT - 1);
        if (shared_face) unpublish<T, N>(pub + (int64_t)old * g.rows + (int64_t)at * N);
        if (tid < parts * GROUP_ND * GROUP_REP) {
            const int h = NP > 1 ? tid / (GROUP_ND * GROUP_REP) : 0,
                      rep = NP > 1 ? tid / GROUP_ND % GROUP_REP : tid / GROUP_ND;
            coherent_store(slots + (((int64_t)rep * GROUP_ROT + old) * GROUP_ND + tid % GROUP_ND) * G + task.rank + h,
                           sentinel_value<double>());
        }
        e++;
        return s_fail == 0;
    };
    // a sum over the group, from its chunks
    auto total = [&](int d) {
        const int q = (e - 1) & 1;
        double s = tot[q][d][0];
#pragma unroll
        for (int c = 1; c < NW / GROUP_ND; c++) s += tot[q][d][c];
        return uniform(s);
    };

    bool ok = true;
    for (;;) {
        Pack<T, N> an[W], a2[W];
        // ---- Ap, (Ap, r*), (r, r)
        const Pack<T, N> Ap = product(p, pn);
        const Pack<T, N> ra = own[1][tid];
        double d2[2] = {0.0, 0.0};
#pragma unroll
        for (int i = 0; i < N; i++) {
            d2[0] = fmadd((double)Ap.v[i], (double)ra.v[i], d2[0]);
            d2[1] = fmadd((double)r.v[i], (double)r.v[i], d2[1]);
        }
        if (!valid) d2[0] = d2[1] = 0.0;
        ok = exchange(Ap, d2, std::integral_constant<int, 2>{}, an);
        if (!ok) break;
        {
            const double D0 = total(0), D1 = total(1);
            resid = uniform(sqrt(D1) / bnorm);
            if (!(resid >= tol) || it >= maxit) {
                done = 1.0;
                break;
            }
            if (brk != 0.0) {
                brk = 0.0;
                restart = 1.0;
                break;
            }
            const double a = uniform(rho / D0);
            if (!(fabs(D0) > 0.0) || !isfinite(a)) {
                restart = 1.0;
                it += 1.0;
                if (it >= maxit) done = 1.0;
                break;
            }
            alpha = a;
            inv_pap = uniform(1.0 / D0);
        }
        const T al = (T)alpha;
        Pack<T, N> s;
#pragma unroll
        for (int i = 0; i < N; i++) s.v[i] = fmadd(-al, Ap.v[i], r.v[i]);
#pragma unroll
        for (int k = 0; k < W; k++)
#pragma unroll
            for (int i = 0; i < N; i++) rn[k].v[i] = fmadd(-al, an[k].v[i], rn[k].v[i]);
        // ---- As, (As, s), (As, As), (As, r*), (s, r*)
        const Pack<T, N> As = product(s, rn);
        const Pack<T, N> rb = own[1][tid];
        double d4[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int i = 0; i < N; i++) {
            const double av = As.v[i], sv = s.v[i], rv = rb.v[i];
            d4[0] = fmadd(av, sv, d4[0]);
            d4[1] = fmadd(av, av, d4[1]);
            d4[2] = fmadd(av, rv, d4[2]);
            d4[3] = fmadd(sv, rv, d4[3]);
        }
        if (!valid) d4[0] = d4[1] = d4[2] = d4[3] = 0.0;
        ok = exchange(As, d4, std::integral_constant<int, 4>{}, a2);
        if (!ok) break;
        {
            const double D[4] = {total(0), total(1), total(2), total(3)};
            // beta = (rho / rho_old) (alpha / omega) with alpha / rho_old = 1 / (r*, Ap)
            const double om = uniform(D[1] > 0 ? D[0] / D[1] : 0.0), inv_om = uniform(D[1] / D[0]);
            const double rn_ = uniform(fmadd(-om, D[2], D[3]));
            omega = om;
            it += 1.0;
            rho_old = rho;
            rho = rn_;
            if (!(fabs(rho) >= eps2 * rast_sq) || om == 0.0) {
                beta = 0.0;
                brk = 1.0;
            } else {
                beta = uniform((rho * inv_pap) * inv_om);
            }
        }
        const T om = (T)omega, be = (T)beta;
        Pack<T, N> x = own[0][tid];
#pragma unroll
        for (int i = 0; i < N; i++) {
            // (n = 1 rounds the other product first: the bits these solves have had)
            x.v[i] += N == 1 ? fmadd(om, s.v[i], al * p.v[i]) : fmadd(al, p.v[i], om * s.v[i]);
            r.v[i] = fmadd(-om, As.v[i], s.v[i]);
            p.v[i] = fmadd(be, fmadd(-om, Ap.v[i], p.v[i]), r.v[i]);
        }
        own[0][tid] = x;
#pragma unroll
        for (int k = 0; k < W; k++)
#pragma unroll
            for (int i = 0; i < N; i++) {
                rn[k].v[i] = fmadd(-om, a2[k].v[i], rn[k].v[i]);
                pn[k].v[i] = fmadd(be, fmadd(-om, an[k].v[i], pn[k].v[i]), rn[k].v[i]);
            }
        if (task.rank == 0 && tid == 0) atomicAdd(g.beat, 1u);
    }
    if (!ok) return false;
    if (valid) {
        st<T, N>(xg + (int64_t)f * N, own[0][tid]);
        st<T, N>(rg + (int64_t)f * N, r);
        st<T, N>(pg + (int64_t)f * N, p);
    }
    if (task.rank == 0 && tid == 0) {
        sc[S_RHO] = rho;
        sc[S_RHO_OLD] = rho_old;
        sc[S_ALPHA] = alpha;
        sc[S_OMEGA] = omega;
        sc[S_BETA] = beta;
        sc[S_RESID] = resid;
        sc[S_IT] = it;
        sc[S_BREAK] = brk;
        sc[S_DONE] = done;
        sc[S_RESTART] = restart;
    }
    return true;
}

#pragma clang fp contract(fast)

// A batch: as many work-groups as fit on the chip at once, each taking share
// after share.  (With one work-group per share, more than fit, the dispatcher
// deals them to the 8 XCDs in turn, an XCD that has got through its eighth stays
// idle, and what is left may not hold all of a segment's shares at once: 11
// instances of 130-163 shares waited for each other until the waits gave up.
// Ten instances of side 230, one step: 55.6-58 -> 32.9 ms; five of side 201:
// 11-33 -> 9.8 ms; 32 ragged ones of 32-192, where no wait gave up: 12.0 -> 11.4 ms.)
template <typename T, int N, int W, int BS, int HOLD, bool BATCH>
__global__ void __launch_bounds__(BS) k_bicg_group(SellView<T> A, GroupView g, T *__restrict__ xg, T *__restrict__ rg,
                                                   T *__restrict__ pg, const T *__restrict__ r_ast,
                                                   const T *__restrict__ qg, T *pub)
{
    do {
    } while (bicg_share<T, N, W, BS, HOLD, BATCH>(A, g, xg, rg, pg, r_ast, qg, pub) && BATCH);
}

// ---------------------------------------------------------------------------
// One cycle of GMRES(m), m <= GMRES_M, in one launch: the same resident groups
// (one segment), left Krylov vectors in the groups' face order, each row read
// and written by its own lane only.  Per iteration three exchanges: the j + 1
// dot products of each of the two Gram-Schmidt passes, then the norm together
// with the unscaled next vector, which the neighbours scale themselves.  The
// Givens rotations are done by one lane of every work-group, the same numbers
// in each.  The launched form takes ten launches and three host reads per
// iteration.  Measured at 197,000 unknowns (20^3 x 6 tetrahedra, n = 2,
// m = 30): 115 -> 24 us per iteration, the step 37.5 -> 7.8 ms (326
// iterations); about 8 us of an iteration are the three exchanges, the rest the
// four passes over V and the rotations.
constexpr int GMRES_M = 32;

struct GmresArgs {
    const double *r0;  // residual
    double *x, *V, *pub;
    int m;
    double beta, bnorm, tol;
    int it, maxit;
};

template <int N, int W, int BS, bool HOLD>
__global__ void __launch_bounds__(BS) k_gmres_group(SellView<double> A, GroupView g, GmresArgs a)
{
    constexpr int NW = BS / 64, MD = GMRES_M / NW, SL = 4;
    __shared__ int s_ticket, s_fail, s_stop;
    __shared__ double part[2][GMRES_M][NW], tot[2][GMRES_M];
    __shared__ Pack<double, N> mine[2][BS];
    __shared__ double H[GMRES_M][GMRES_M], hc[GMRES_M + 1], cs[GMRES_M], sn[GMRES_M], gv[GMRES_M + 1], ys[GMRES_M];
    const int tid = threadIdx.x, lane = tid & 63, wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    if (tid == 0) {
        s_ticket = atomicAdd(g.ticket, 1);
        s_fail = 0;
        s_stop = 0;
        gv[0] = a.beta;
    }
    __syncthreads();
    const int ticket = __builtin_amdgcn_readfirstlane(s_ticket);
    if (ticket >= g.total) return;
    const GroupTask task = g.task[ticket];
    double *sc = g.sc;
    const int G = g.seg[0].y;
    double *slots = g.slots;
    const int at = task.p0 + tid;
    const bool valid = at < task.p1;
    const int f = valid ? g.face[at] : 0;

    int col[W];
    Pack<double, N * N> val[HOLD ? W : 1];
    Pack<double, (N > 1 ? N * (N - 1) : 1)> dg;
    Pack<double, N> v, vn[W];
    int w = 0;
#pragma unroll
    for (int i = 0; i < N; i++) v.v[i] = 0.0;
    if constexpr (N > 1) {
#pragma unroll
        for (int i = 0; i < N * (N - 1); i++) dg.v[i] = 0.0;
    }
    int64_t base = 0;
    if (valid) {
        base = A.slice_ptr[f >> 6] + (f & 63);
        w = A.slice_width[f >> 6];
    }
    const double inv0 = 1.0 / a.beta;
    unsigned remote = 0;
    bool alone = true;
#pragma unroll
    for (int k = 0; k < W; k++) {
        col[k] = k < w ? A.col[base + (int64_t)k * 64] : f;
        if constexpr (HOLD) {
#pragma unroll
            for (int i = 0; i < N * N; i++) val[k].v[i] = 0.0;
        }
#pragma unroll
        for (int i = 0; i < N; i++) vn[k].v[i] = 0.0;
        if (k < w) {
            if constexpr (HOLD) val[k] = ld<double, N * N>(A.val + (base + (int64_t)k * 64) * (N * N));
            vn[k] = ld<double, N>(a.r0 + (int64_t)col[k] * N);
#pragma unroll
            for (int i = 0; i < N; i++) vn[k].v[i] *= inv0;
        }
        alone = alone && col[k] == f;
        col[k] = k < w ? g.pos[col[k]] : task.p0;
        if (col[k] < task.p0 || col[k] >= task.p1) remote |= 1u << k;
        else col[k] = -1 - (col[k] - task.p0);
    }
    const bool shared_face = valid && (remote != 0 || alone);
    if (valid) {
        v = ld<double, N>(a.r0 + (int64_t)f * N);
#pragma unroll
        for (int i = 0; i < N; i++) v.v[i] *= inv0;
        if constexpr (N > 1) dg = ld<double, N *(N - 1)>(A.val + A.diag_base + (int64_t)f * N * (N - 1));
    }
    GroupWait wait(g, sc + S_FAIL);
    int e = 0, pe = 0, posted = 0;  // reductions, publications, dot products of the last reduction
    Pack<double, N> wv, wn[W];

    // the sums over the group of part[e & 1][0..nd) into tot[e & 1]; with
    // PUB the publication of wv and the neighbours' values into wn
    auto reduce = [&](int nd, auto PUBC) {
        constexpr bool PUB = decltype(PUBC)::value;
        const int rot = e & (GROUP_ROT - 1), par = e & 1;
        double *pb = a.pub + (int64_t)(pe & (GROUP_ROT - 1)) * g.rows;
        if constexpr (PUB) {
            if (shared_face) publish<double, N>(pb + (int64_t)at * N, wv);
            mine[pe & 1][tid] = wv;
        }
        __syncthreads();
        if (tid < nd) {
            double s = part[par][tid][0];
#pragma unroll
            for (int q = 1; q < NW; q++) s += part[par][tid][q];
            if (is_sentinel(s)) s = __builtin_nan("");
            coherent_store(slots + ((int64_t)rot * GMRES_M + tid) * G + task.rank, s);
        }
        unsigned pend = 0, pd = 0;
        if constexpr (PUB) {
            pend = remote;
#pragma unroll
            for (int k = 0; k < W; k++)
                if (col[k] < 0) wn[k] = mine[pe & 1][-1 - col[k]];
        }
        // wave q adds the dots q, q + NW, ...
        double s4[MD][SL];
#pragma unroll
        for (int d = 0; d < MD; d++)
#pragma unroll
            for (int q = 0; q < SL; q++) {
                s4[d][q] = 0.0;
                if (wid + NW * d < nd && q * 64 + lane < G) pd |= 1u << (d * SL + q);
            }
        __builtin_amdgcn_s_sleep(GROUP_FIRST_LOOK);
        for (;;) {
            if constexpr (PUB) {
#pragma unroll
                for (int k = 0; k < W; k++)
                    if (pend >> k & 1u) wn[k] = look<double, N>(pb + (int64_t)col[k] * N);
            }
#pragma unroll
            for (int d = 0; d < MD; d++)
#pragma unroll
                for (int q = 0; q < SL; q++)
                    if (pd >> (d * SL + q) & 1u)
                        s4[d][q] = coherent_load(slots + ((int64_t)rot * GMRES_M + wid + NW * d) * G + q * 64 + lane);
            if constexpr (PUB) {
#pragma unroll
                for (int k = 0; k < W; k++) {
                    bool there = true;
#pragma unroll
                    for (int i = 0; i < N; i++) there = there && !is_sentinel(wn[k].v[i]);
                    if (there) pend &= ~(1u << k);
                }
            }
#pragma unroll
            for (int d = 0; d < MD; d++)
#pragma unroll
                for (int q = 0; q < SL; q++)
                    if (!is_sentinel(s4[d][q])) pd &= ~(1u << (d * SL + q));
            if (!__any((pend | pd) != 0)) break;
            if (wait.pause()) {
                if (lane == 0) s_fail = 1;
                break;
            }
        }
        wait.t0 = 0;
#pragma unroll
        for (int d = 0; d < MD; d++)
            if (wid + NW * d < nd) {
                const double one[1] = {(s4[d][0] + s4[d][1]) + (s4[d][2] + s4[d][3])};
                const double s = sums_wave<1>(one);
                if (lane == 0) tot[par][wid + NW * d] = s;
            }
        memory_done();
        __syncthreads();
        // all have posted this reduction, so the sums of the previous one and
        // (PUB) the previous publication have been read
        if (tid < posted)
            coherent_store(slots + ((int64_t)((e + GROUP_ROT - 1) & (GROUP_ROT - 1)) * GMRES_M + tid) * G + task.rank,
                           sentinel_value<double>());
        if constexpr (PUB) {
            if (shared_face)
                unpublish<double, N>(a.pub + (int64_t)((pe + GROUP_ROT - 1) & (GROUP_ROT - 1)) * g.rows +
                                     (int64_t)at * N);
            pe++;
        }
        posted = nd;
        e++;
        return s_fail == 0;
    };

    double *const Vr = a.V + (int64_t)(valid ? at : 0) * N;  // this lane's rows
    int j = 0, it = a.it;
    bool ok = true;
    for (; j < a.m && it < a.maxit; j++) {
        if (valid) st<double, N>(Vr + (int64_t)j * g.rows, v);
        // w = A v
        wv = v;
        if constexpr (N > 1) {
#pragma unroll
            for (int i = 0; i < N; i++)
#pragma unroll
                for (int q = 0; q < N; q++)
                    if (q != i) wv.v[i] += dg.v[i * (N - 1) + (q < i ? q : q - 1)] * v.v[q];
        }
#pragma unroll
        for (int k = 0; k < W; k++) {
            if constexpr (!HOLD) {
                if (k < w) val[0] = ld<double, N * N>(A.val + (base + (int64_t)k * 64) * (N * N));
            }
            if (HOLD || k < w) {
#pragma unroll
                for (int i = 0; i < N; i++)
#pragma unroll
                    for (int q = 0; q < N; q++) wv.v[i] += val[HOLD ? k : 0].v[i * N + q] * vn[k].v[q];
            }
        }
        // classical Gram-Schmidt, twice
        for (int pass = 0; pass < 2 && ok; pass++) {
            for (int k0 = 0; k0 <= j; k0 += 4) {
                double d4[4] = {0.0, 0.0, 0.0, 0.0};
                if (valid) {
                    Pack<double, N> q4[4];
#pragma unroll
                    for (int q = 0; q < 4; q++) q4[q] = ld<double, N>(Vr + (int64_t)min(k0 + q, j) * g.rows);
#pragma unroll
                    for (int q = 0; q < 4; q++)
#pragma unroll
                        for (int i = 0; i < N; i++) d4[q] += q4[q].v[i] * wv.v[i];
                }
                const double s = sums_wave<4>(d4);
                // (dots past j repeat dot j and are not read)
                if ((lane & 15) == 0) part[e & 1][k0 + (lane >> 4)][wid] = s;
            }
            ok = reduce(j + 1, std::false_type{});
            const double *t = tot[(e - 1) & 1];
            if (tid <= j) hc[tid] = pass ? hc[tid] + t[tid] : t[tid];
            for (int k0 = 0; k0 <= j; k0 += 4) {
                if (valid) {
                    Pack<double, N> q4[4];
#pragma unroll
                    for (int q = 0; q < 4; q++) q4[q] = ld<double, N>(Vr + (int64_t)min(k0 + q, j) * g.rows);
#pragma unroll
                    for (int q = 0; q < 4; q++) {
                        const double h = k0 + q <= j ? t[k0 + q] : 0.0;
#pragma unroll
                        for (int i = 0; i < N; i++) wv.v[i] -= h * q4[q].v[i];
                    }
                }
            }
        }
        if (!ok) break;
        double n2[1] = {0.0};
        if (valid) {
#pragma unroll
            for (int i = 0; i < N; i++) n2[0] += wv.v[i] * wv.v[i];
        }
        const double s = sums_wave<1>(n2);
        if (lane == 0) part[e & 1][0][wid] = s;
        ok = reduce(1, std::true_type{});
        if (!ok) break;
        const double hn = sqrt(uniform(tot[(e - 1) & 1][0]));
        it++;
        if (tid == 0) {
            // the earlier rotations, then the one that clears hn
            double h = hc[0];
            for (int q = 0; q < j; q++) {
                const double h1 = hc[q + 1], c = cs[q], d = sn[q];
                H[q][j] = c * h + d * h1;
                h = -d * h + c * h1;
            }
            const double den = sqrt(h * h + hn * hn);
            const double c = den > 0 ? h / den : 1.0, d = den > 0 ? hn / den : 0.0;
            cs[j] = c;
            sn[j] = d;
            H[j][j] = c * h + d * hn;
            gv[j + 1] = -d * gv[j];
            gv[j] = c * gv[j];
            const double resid = fabs(gv[j + 1]) / a.bnorm;
            if (resid < a.tol) s_stop = 1;
            if (task.rank == 0) {
                sc[S_RESID] = resid;
                sc[S_IT] = it;
                atomicAdd(g.beat, 1u);
            }
        }
        __syncthreads();
        const double inv = 1.0 / hn;
#pragma unroll
        for (int i = 0; i < N; i++) v.v[i] = wv.v[i] * inv;
#pragma unroll
        for (int k = 0; k < W; k++)
#pragma unroll
            for (int i = 0; i < N; i++) vn[k].v[i] = wn[k].v[i] * inv;
        if (s_stop) {
            j++;
            break;
        }
    }
    if (!ok) return;
    // y from the triangular system, x += V y
    if (tid == 0) {
        for (int q = j - 1; q >= 0; q--) {
            double s = gv[q];
            for (int t = q + 1; t < j; t++) s -= H[q][t] * ys[t];
            ys[q] = s / H[q][q];
        }
    }
    __syncthreads();
    if (valid) {
        Pack<double, N> s;
#pragma unroll
        for (int i = 0; i < N; i++) s.v[i] = 0.0;
        for (int k = 0; k < j; k++) {
            const Pack<double, N> q = ld<double, N>(Vr + (int64_t)k * g.rows);
#pragma unroll
            for (int i = 0; i < N; i++) s.v[i] += ys[k] * q.v[i];
        }
        Pack<double, N> x = ld<double, N>(a.x + (int64_t)f * N);
#pragma unroll
        for (int i = 0; i < N; i++) x.v[i] += s.v[i];
        st<double, N>(a.x + (int64_t)f * N, x);
    }
}

// sentinels in the published vectors and the slots, counters at zero; where
// the segment (sc) has stopped already, the counters only
template <typename T>
__global__ void __launch_bounds__(256) k_group_prepare(int64_t pubn, T *pub, int slotn, double *slots, int *ticket,
                                                       unsigned *beat, const double *sc)
{
    const int64_t stride = (int64_t)gridDim.x * 256, t = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (sc && halted(sc)) pubn = slotn = 0;
    for (int64_t i = t; i < pubn; i += stride) pub[i] = sentinel_value<T>();
    for (int64_t i = t; i < slotn; i += stride) slots[i] = sentinel_value<double>();
    if (t == 0) {
        *ticket = 0;
        *beat = 0;
    }
}

// segments whose waits gave up: the host restarts them from their iterate
__global__ void k_group_failed(double *sc, int nseg)
{
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= nseg) return;
    double *q = sc + (int64_t)s * NSLOTS;
    if (q[S_FAIL] != 0.0) {
        q[S_FAIL] = 0.0;
        q[S_DONE] = 0.0;
        q[S_RESTART] = 1.0;
    }
}

namespace {

template <typename F>
void with_shape(int n, int width, F &&f)
{
    auto go = [&](auto NC) {
        if (width <= 4) f(NC, std::integral_constant<int, 4>{});
        else if (width <= 6) f(NC, std::integral_constant<int, 6>{});
        else f(NC, std::integral_constant<int, 10>{});
    };
    if (n == 1) go(std::integral_constant<int, 1>{});
    else if (n == 2) go(std::integral_constant<int, 2>{});
    else go(std::integral_constant<int, 3>{});
}
// Registers of a lane, about: a work-group of 1024 threads has 128, of 512
// 256, of 256 512 (part of them accumulation registers).  Shapes past 400
// do not hold the matrix in registers.
constexpr int lane_registers(int bytes, int n, int w) { return bytes / 4 * (n * (4 * w + 7) + n * n * (w + 1)) + w + 30; }
constexpr int max_threads(int bytes, int n, int w)
{
    return lane_registers(bytes, n, w) <= 92 ? 1024 : lane_registers(bytes, n, w) <= 240 ? 512 : 256;
}
constexpr bool holds(int bytes, int n, int w) { return lane_registers(bytes, n, w) <= 400; }
// f(the way the matrix rows are held): registers where they fit, else LDS (when
// the plan gives a work-group at most LDS_FACES faces) or memory
template <typename T, int N, int W, typename F>
void with_hold(bool lds, F &&f)
{
    if constexpr (holds(sizeof(T), N, W)) f(std::integral_constant<int, HOLD_REGS>{});
    else if (lds) f(std::integral_constant<int, HOLD_LDS>{});
    else f(std::integral_constant<int, HOLD_MEMORY>{});
}
template <typename T, typename F>
void with_threads(int bs, int n, int w, F &&f)
{
    with_shape(n, w, [&](auto NC, auto WC) {
        constexpr int M = max_threads(sizeof(T), decltype(NC)::value, decltype(WC)::value);
        if constexpr (M == 1024)
            if (bs == 1024) return f(NC, WC, std::integral_constant<int, 1024>{});
        f(NC, WC, std::integral_constant<int, (M < 512 ? M : 512)>{});
    });
}

constexpr int BATCH_WIDTH = 6;
// f(the BiCGStab kernel, its threads); batches are FP64 and on simplices
template <typename T, typename F>
void with_bicg_group(int bs, int n, int width, bool lds, bool batch, F &&f)
{
    with_threads<T>(bs, n, width, [&](auto NC, auto WC, auto BC) {
        constexpr int N = decltype(NC)::value, W = decltype(WC)::value, BS = decltype(BC)::value;
        with_hold<T, N, W>(lds, [&](auto HC) {
            constexpr int HOLD = decltype(HC)::value;
            if constexpr (sizeof(T) == 8 && W <= BATCH_WIDTH)
                if (batch) return f(&k_bicg_group<T, N, W, BS, HOLD, true>, BS);
            f(&k_bicg_group<T, N, W, BS, HOLD, false>, BS);
        });
    });
}

// The faces of every segment in Morton order of their positions (the lowest
// corner of the first cell: a cell's faces stay together), so that a
// work-group's faces are a compact piece of the mesh and few of their
// neighbours belong to other work-groups.  Stable, by a radix sort of 33 bits.
void group_order(const Ctx &c, std::vector<int> &face)
{
    for (int E = 0; E < c.F; E++) face[E] = E;
    if (c.h_face_pos.size() != 3 * (size_t)c.F) return;
    std::vector<uint64_t> key, other;
    for (size_t s = 0; s + 1 < c.h_seg_faces.size(); s++) {
        const int f0 = c.h_seg_faces[s], F = c.h_seg_faces[s + 1] - f0;
        if (F < 2) continue;
        const float *p = c.h_face_pos.data() + 3 * (size_t)f0;
        float lo[3], hi[3], scale[3];
        for (int d = 0; d < 3; d++) lo[d] = hi[d] = p[d];
        for (int E = 0; E < F; E++)
            for (int d = 0; d < 3; d++) {
                lo[d] = std::min(lo[d], p[3 * (size_t)E + d]);
                hi[d] = std::max(hi[d], p[3 * (size_t)E + d]);
            }
        for (int d = 0; d < 3; d++) scale[d] = hi[d] > lo[d] ? 2047.0f / (hi[d] - lo[d]) : 0.0f;
        // bits 32.., the key; below, the face
        auto spread = [](uint64_t v) {  // 11 bits to every third bit
            v = (v | v << 16) & 0x30000ffull;
            v = (v | v << 8) & 0x300f00full;
            v = (v | v << 4) & 0x30c30c3ull;
            return (v | v << 2) & 0x9249249ull;
        };
        key.resize(F);
        other.resize(F);
        for (int E = 0; E < F; E++) {
            uint64_t m = 0;
            for (int d = 0; d < 3; d++) {
                const uint64_t q = (uint64_t)std::min(2047.0f, std::max(0.0f, (p[3 * (size_t)E + d] - lo[d]) * scale[d]));
                m |= (spread(q & 1023) | (q >> 10) << 30) << d;
            }
            key[E] = m << 31 | (uint64_t)E;
        }
        for (int pass = 0; pass < 3; pass++) {
            std::vector<int> count(2049, 0);
            const int shift = 31 + 11 * pass;
            for (int E = 0; E < F; E++) count[((key[E] >> shift) & 2047) + 1]++;
            for (int b = 0; b < 2048; b++) count[b + 1] += count[b];
            for (int E = 0; E < F; E++) other[count[(key[E] >> shift) & 2047]++] = key[E];
            key.swap(other);
        }
        for (int E = 0; E < F; E++) face[f0 + E] = f0 + (int)(key[E] & 0x7fffffffull);
    }
}

}  // namespace

bool group_plan(Ctx &c, GroupPlan &gp, bool fp32, int width, bool gmres, const std::vector<int> &iperm)
{
    gp.total = 0;
    if (width > 10 || width < 1) return false;
    const int cap_bs = [&] {
        int m = 256;
        with_shape(c.n, width, [&](auto NC, auto WC) {
            m = max_threads(fp32 ? 4 : 8, decltype(NC)::value, decltype(WC)::value);
        });
        return m;
    }();
    int cus = 0;
    MHFEM_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, c.device));
    const int nseg = (int)c.h_seg_faces.size() - 1;
    if (nseg > 1 && width > BATCH_WIDTH) return false;
    bool regs = true;
    with_shape(c.n, width, [&](auto NC, auto WC) {
        regs = holds(gmres || !fp32 ? 8 : 4, decltype(NC)::value, decltype(WC)::value);
    });
    // Faces of a part, at most, by the faces of its segment alone: an instance
    // is summed in a batch as in a context of its own.  Rows that do not fit
    // in registers are held in LDS while one work-group of LDS_FACES faces per
    // CU holds the segment (20^3 voxels n = 3: 16.5 -> 9.7 us per iteration; a
    // product took 3.5 us from the L2).
    auto most = [&](int F) {
        return !regs && !gmres && F <= LDS_FACES * cus ? LDS_FACES : part_threads(cap_bs);
    };
    auto split = [&](int F, int &G, int &part) {
        G = std::max(1, (F + most(F) - 1) / most(F));
        part = std::min(most(F), ((F + G - 1) / G + 63) / 64 * 64);
        G = std::max(1, (F + part - 1) / std::max(1, part));
    };
    // 512 threads while one such work-group per CU holds every face (64 x 64
    // x 2 triangles: 0.63 ms with 512, 0.76 ms with 1024); more faces take the
    // largest the registers allow (32 ragged instances, 1.5 M faces: 16.7 ms
    // with 512 and two work-groups per CU, 11.4 with 1024)
    const int bs = gmres || c.F <= 512 * cus ? std::min(512, cap_bs) : cap_bs, np = bs / part_threads(bs);
    // the segments whose shares fit on the chip at once are planned; the
    // others of a batch iterate by launches afterwards
    bool lds = !regs && !gmres;
    const int cap = std::min(cus, 256);
    std::vector<int> order;
    for (int s = 0; s < nseg; s++) {
        const int F = c.h_seg_faces[s + 1] - c.h_seg_faces[s];
        int G, part;
        split(F, G, part);
        if ((G + np - 1) / np > cap) continue;
        order.push_back(s);
        lds = lds && F <= LDS_FACES * cus;
    }
    if (order.empty()) return false;
    int per_cu = 0;
    auto occupancy = [&](auto *kernel, int threads) {
        MHFEM_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, threads, 0));
    };
    if (gmres)
        with_threads<double>(bs, c.n, width, [&](auto NC, auto WC, auto BC) {
            constexpr int N = decltype(NC)::value, W = decltype(WC)::value, BS = std::min(512, decltype(BC)::value);
            occupancy(k_gmres_group<N, W, BS, holds(8, N, W)>, BS);
        });
    else if (fp32) with_bicg_group<float>(bs, c.n, width, lds, nseg > 1, occupancy);
    else with_bicg_group<double>(bs, c.n, width, lds, nseg > 1, occupancy);
    if (per_cu < 1) return false;
    std::vector<GroupTask> tasks;
    std::vector<int2> segs(nseg, int2{0, 0});
    std::stable_sort(order.begin(), order.end(), [&](int a, int b) {
        return c.h_seg_faces[a + 1] - c.h_seg_faces[a] > c.h_seg_faces[b + 1] - c.h_seg_faces[b];
    });
    // positions: each segment's faces along a space-filling curve
    std::vector<int> face(c.F), pos(c.F);
    group_order(c, face);
    long slot = 0;
    for (int s : order) {
        const int f0 = c.h_seg_faces[s], F = c.h_seg_faces[s + 1] - f0;
        int G, part;
        split(F, G, part);
        segs[s] = int2{(int)slot, G};
        slot += gmres ? (long)GROUP_ROT * GMRES_M * G : (long)GROUP_REP * GROUP_ROT * GROUP_ND * G;
        for (int q = 0; q < G; q += np)
            tasks.push_back(GroupTask{s, q, f0 + q * part, std::min(f0 + F, f0 + (q + np) * part), part});
    }
    gp.threads = bs;
    gp.resident = per_cu * cus;
    gp.batch = nseg > 1;
    gp.lds = lds;
    gp.hold = regs ? HOLD_REGS : lds ? HOLD_LDS : HOLD_MEMORY;
    gp.width = width;
    gp.total = (int)tasks.size();
    gp.nslots = (int)slot;
    gp.task.alloc(tasks.size());
    auto tables = [&](DBuf<int> &df, DBuf<int> &dp) {
        for (int q = 0; q < c.F; q++) pos[face[q]] = q;
        df.alloc(c.F);
        dp.alloc(c.F);
        MHFEM_HIP(hipMemcpy(df.p, face.data(), c.F * sizeof(int), hipMemcpyHostToDevice));
        MHFEM_HIP(hipMemcpy(dp.p, pos.data(), c.F * sizeof(int), hipMemcpyHostToDevice));
    };
    tables(gp.face, gp.pos);
    if (!iperm.empty()) {
        // the same places on the curve, whatever the copy's numbers (us per
        // iteration with the curve laid over the copy's numbers -> over the
        // faces: 20^3 x 6 tetrahedra, n = 1, 6.2 -> 5.7; n = 2, FP32, 8.1 -> 7.7;
        // 20^3 voxels, n = 3, 12.7 -> 10.8; neighbours in other work-groups
        // 90 % -> 16 % at 12^3 x 6)
        for (int q = 0; q < c.F; q++) face[q] = iperm[face[q]];
        tables(gp.face_p, gp.pos_p);
    }
    gp.seg.alloc(2 * (size_t)nseg);
    MHFEM_HIP(hipMemcpy(gp.task.p, tasks.data(), tasks.size() * sizeof(GroupTask), hipMemcpyHostToDevice));
    MHFEM_HIP(hipMemcpy(gp.seg.p, segs.data(), segs.size() * sizeof(int2), hipMemcpyHostToDevice));
    gp.slots.alloc(slot);
    gp.counters.alloc(2);
    gp.pub.alloc((size_t)GROUP_ROT * c.rows * (fp32 ? 4 : 8));
    return true;
}

template <typename T>
void group_iterate(Ctx &c, GroupPlan &gp, const SellView<T> &A, bool permuted, double *sc, T *x, T *r, T *p,
                   const T *r_ast, const T *q)
{
    const int *face = permuted ? gp.face_p.p : gp.face.p, *pos = permuted ? gp.pos_p.p : gp.pos.p;
    gp.launches++;
    gp.slice_ptr = A.slice_ptr;
    gp.slice_width = A.slice_width;
    gp.col = A.col;
    gp.last_pos = pos;
    const int64_t pubn = (int64_t)GROUP_ROT * c.rows;
    T *pub = reinterpret_cast<T *>(gp.pub.p);
    int *ticket = gp.counters.p;
    unsigned *beat = reinterpret_cast<unsigned *>(gp.counters.p + 1);
    const unsigned g = (unsigned)std::min<int64_t>(1024, (std::max<int64_t>(pubn, gp.nslots) + 255) / 256);
    hipLaunchKernelGGL(k_group_prepare<T>, g, 256, 0, c.stream, pubn, pub, gp.nslots, gp.slots.p, ticket, beat,
                       q ? (const double *)sc : (const double *)nullptr);
    const GroupView v{gp.total, c.rows, gp.task.p, face, pos, reinterpret_cast<const int2 *>(gp.seg.p),
                      ticket, beat, gp.slots.p, sc, gp.wait_ticks};
    with_bicg_group<T>(gp.threads, c.n, gp.width, gp.lds, gp.batch, [&](auto *kernel, int threads) {
        hipLaunchKernelGGL(kernel, std::min(gp.total, gp.resident), threads, 0, c.stream, A, v, x, r, p, r_ast, q, pub);
    });
    MHFEM_HIP(hipGetLastError());
}
template void group_iterate<double>(Ctx &, GroupPlan &, const SellView<double> &, bool, double *, double *, double *,
                                    double *, const double *, const double *);
template void group_iterate<float>(Ctx &, GroupPlan &, const SellView<float> &, bool, double *, float *, float *, float *,
                                   const float *, const float *);

int group_gmres_restart() { return GMRES_M; }

void group_gmres_cycle(Ctx &c, GroupPlan &gp, const SellView<double> &A, double *sc, const double *r, double *x,
                       double *V, int m, double beta, double bnorm, double tol, int it, int maxit)
{
    gp.launches++;
    gp.slice_ptr = A.slice_ptr;
    gp.slice_width = A.slice_width;
    gp.col = A.col;
    gp.last_pos = gp.pos.p;
    const int64_t pubn = (int64_t)GROUP_ROT * c.rows;
    double *pub = reinterpret_cast<double *>(gp.pub.p);
    int *ticket = gp.counters.p;
    unsigned *beat = reinterpret_cast<unsigned *>(gp.counters.p + 1);
    const unsigned g = (unsigned)std::min<int64_t>(1024, (std::max<int64_t>(pubn, gp.nslots) + 255) / 256);
    hipLaunchKernelGGL(k_group_prepare<double>, g, 256, 0, c.stream, pubn, pub, gp.nslots, gp.slots.p, ticket, beat,
                       (const double *)nullptr);
    const GroupView v{gp.total, c.rows, gp.task.p, gp.face.p, gp.pos.p, reinterpret_cast<const int2 *>(gp.seg.p),
                      ticket, beat, gp.slots.p, sc, gp.wait_ticks};
    const GmresArgs a{r, x, V, pub, m, beta, bnorm, tol, it, maxit};
    with_threads<double>(gp.threads, c.n, gp.width, [&](auto NC, auto WC, auto BC) {
        constexpr int N = decltype(NC)::value, W = decltype(WC)::value, BS = std::min(512, decltype(BC)::value);
        hipLaunchKernelGGL((k_gmres_group<N, W, BS, holds(8, N, W)>), gp.total, BS, 0, c.stream, A, v, a);
    });
    MHFEM_HIP(hipGetLastError());
}

void group_last(Ctx &c, GroupPlan &gp, long long *iterations, long long *neighbours, long long *remote)
{
    *iterations = *neighbours = *remote = 0;
    if (!gp.launches) return;
    MHFEM_HIP(hipStreamSynchronize(c.stream));
    const int slices = (c.F + 63) / 64;
    std::vector<int64_t> ptr(slices);
    std::vector<int> width(slices), pos(c.F), col;
    std::vector<GroupTask> task(gp.total);
    unsigned beat = 0;
    auto get = [](auto *dst, const void *src, size_t count) {
        MHFEM_HIP(hipMemcpy(dst, src, count * sizeof(*dst), hipMemcpyDeviceToHost));
    };
    get(&beat, gp.counters.p + 1, 1);
    get(ptr.data(), gp.slice_ptr, ptr.size());
    get(width.data(), gp.slice_width, width.size());
    get(pos.data(), gp.last_pos, pos.size());
    get(task.data(), gp.task.p, task.size());
    col.resize((size_t)ptr[slices - 1] + 64 * (size_t)width[slices - 1]);
    get(col.data(), gp.col, col.size());
    std::vector<int> group(c.F, -1);  // by position
    for (size_t q = 0; q < task.size(); q++)
        for (int at = task[q].p0; at < task[q].p1; at++) group[at] = (int)q;
    for (int f = 0; f < c.F; f++)
        for (int k = 0; k < width[f / 64]; k++) {
            const int to = col[(size_t)ptr[f / 64] + 64 * (size_t)k + f % 64];
            if (to == f) continue;  // padding
            ++*neighbours;
            *remote += group[pos[to]] != group[pos[f]];
        }
    *iterations = beat;
}

void group_clear_failed(Ctx &c, double *sc, int nseg)
{
    hipLaunchKernelGGL(k_group_failed, (nseg + 63) / 64, 64, 0, c.stream, sc, nseg);
    MHFEM_HIP(hipGetLastError());
}

}  // namespace mhfem
