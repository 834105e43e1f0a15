// Kernels of the multigrid levels that are not marched plane by plane: the levels below
// 128 cells a side under a finer one, every 2D level and the small 3D grids, and the
// fused cycle of the coarsest levels.
//
// These levels fit the caches, and what bounds a pass on them is the number of vector
// instructions (a wave64 instruction holds a CDNA SIMD for four cycles) and the latency
// of one dependent chain, not bytes.  So nodes are addressed by a 32-bit offset from
// per-field scalar bases, index splits are shifts (every level side is a power of two)
// and each lane does useful work (a colour pass has one lane per pair of cells, one of
// each colour).  The arithmetic is that of the per-node kernels of st_kernels.hip in
// the same order (st_box.h).
//
// Against the kernels with 64-bit indices, a lane per node and range tests per access,
// us per launch in FP64 / FP32: colour pass 64^3 23.7 / 17.2 -> 9.9 / 7.8, 32^3 9.5 / 8.3
// -> 4.6 / 4.3, 16^3 8.9 / 7.8 -> 4.4 / 4.2, 2D 256^2 FP32 6.9 -> 5.7 (finest level),
// 64^2 6.4 -> 3.6; residual and restriction 32^3 7.4 + 4.9 -> 7.8 in one launch, 64^2 FP32
// 4.3 + 3.6 -> 3.9.  About 3 us of each is the launch and one trip to memory.
#include "st_box.h"
#include "st_kernels.h"

namespace st {

// ------------------------------------------------------------ colour pass

// One colour of the smoother, xin -> xout, one lane per pair of cells along the fastest
// axis: the lane solves the block of the pair's colour cell and copies what the colour
// does not own (the other cell's p, and its faces on the domain boundary).  lg: log2 of
// the level side.  ZERO: xin is zero and not read.
template <typename TS, int DIM, bool ZERO, bool MASK, bool FINE>
__global__ void __launch_bounds__(256) k_box(Lvl g, int lg, const uint8_t *__restrict__ fl, const TS *__restrict__ al,
                                             const TS *__restrict__ b, const TS *__restrict__ xin,
                                             TS *__restrict__ xout, int color, float omega)
{
    typedef typename Cvt<TS>::C C;
    const unsigned t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (1u << (DIM * lg - 1))) return;
    const int m = (1 << lg) - 1;
    const int pr = (int)(t & (unsigned)(m >> 1)) * 2;  // even cell of the pair along the fastest axis
    int i, j, k, oj, ok;                               // the colour cell; (i, oj, ok) the other one
    if (DIM == 3) {
        j = oj = (int)(t >> (lg - 1)) & m;
        i = (int)(t >> (2 * lg - 1));
        k = pr + ((i + j + color) & 1);
        ok = 2 * pr + 1 - k;
    } else {
        i = (int)(t >> (lg - 1));
        j = pr + ((i + color) & 1);
        oj = 2 * pr + 1 - j;
        k = ok = 0;
    }
    const CellAcc<TS, DIM, MASK> a(g, fl, al, b, xin, i, j, k);
    C pn, u0[3], u1[3];
    box_cell<C, DIM, ZERO, FINE>(a, omega, pn, u0, u1);
    const long st[3] = {a.sI, a.sJ, 1};
    // copy-through first (its loads are independent of the solve)
    const unsigned qo = a.q + (DIM == 3 ? (unsigned)(ok - k) : (unsigned)(oj - j));
    auto cp = [&](int f, long off) {
        TS v;
        if (ZERO) v = Cvt<TS>::st(C(0));
        else v = at(xin + f * g.S + off, qo);
        put(xout + f * g.S + off, qo, v);
    };
    cp(0, 0);
    if (i == 0) cp(1, 0);
    if (i == g.nx - 1) cp(1, st[0]);
    if (oj == 0) cp(2, 0);
    if (oj == g.ny - 1) cp(2, st[1]);
    if (DIM == 3) {
        if (ok == 0) cp(3, 0);
        if (ok == g.nz - 1) cp(3, st[2]);
    }
    put(xout, a.q, Cvt<TS>::st(pn));
#pragma unroll
    for (int d = 0; d < DIM; d++) {
        put(xout + (1 + d) * g.S, a.q, Cvt<TS>::st(u0[d]));
        put(xout + (1 + d) * g.S + st[d], a.q, Cvt<TS>::st(u1[d]));
    }
}

// ------------------------------------------------------ operator, residual

// node of a linear index over the padded box (rows of Pz)
template <int DIM> __device__ __forceinline__ void box_node(const Lvl &g, unsigned n, int &i, int &j, int &k)
{
    if (DIM == 3) {
        const unsigned t = n / (unsigned)g.Pz;
        k = (int)(n - t * (unsigned)g.Pz);
        i = (int)(t / (unsigned)g.Py);
        j = (int)(t - (unsigned)i * (unsigned)g.Py);
    } else {
        i = (int)(n / (unsigned)g.Py);
        j = (int)(n - (unsigned)i * (unsigned)g.Py);
        k = 0;
    }
}

// y = A x, one node per lane (these levels have no row padding)
template <typename TS, int DIM>
__global__ void __launch_bounds__(256) k_apply(Lvl g, const uint8_t *__restrict__ fl, const TS *__restrict__ al,
                                               const TS *__restrict__ x, TS *__restrict__ y)
{
    typedef typename Cvt<TS>::C C;
    const unsigned n = blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= (unsigned)g.S) return;
    int i, j, k;
    box_node<DIM>(g, n, i, j, k);
    const NodeAcc<TS, DIM, true> a(g, fl, al, x, i, j, k);
    const BoxSten<C, DIM, NodeAcc<TS, DIM, true>> s{a};
    put(y, n, Cvt<TS>::st(s.cell()));
    put(y + g.S, n, Cvt<TS>::st(s.template face<0>(0, 0, 0)));
    put(y + 2 * g.S, n, Cvt<TS>::st(s.template face<1>(0, 0, 0)));
    if (DIM == 3) put(y + 3 * g.S, n, Cvt<TS>::st(s.template face<2>(0, 0, 0)));
}

// r = b - A x (without r: the norm only), and the block's partial sum of |r|^2
template <typename TS, int DIM>
__global__ void __launch_bounds__(256) k_residual(Lvl g, const uint8_t *__restrict__ fl, const TS *__restrict__ al,
                                                  const TS *__restrict__ b, const TS *__restrict__ x, TS *r,
                                                  double *part)
{
    typedef typename Cvt<TS>::C C;
    __shared__ double sh[4];
    const unsigned n = blockIdx.x * blockDim.x + threadIdx.x;
    double acc = 0.0;
    if (n < (unsigned)g.S) {
        int i, j, k;
        box_node<DIM>(g, n, i, j, k);
        const NodeAcc<TS, DIM, true> a(g, fl, al, x, i, j, k);
        const BoxSten<C, DIM, NodeAcc<TS, DIM, true>> s{a};
        C v[4];
        v[0] = Cvt<TS>::ld(at(b, n)) - s.cell();
        v[1] = Cvt<TS>::ld(at(b + g.S, n)) - s.template face<0>(0, 0, 0);
        v[2] = Cvt<TS>::ld(at(b + 2 * g.S, n)) - s.template face<1>(0, 0, 0);
        if (DIM == 3) v[3] = Cvt<TS>::ld(at(b + 3 * g.S, n)) - s.template face<2>(0, 0, 0);
#pragma unroll
        for (int f = 0; f <= DIM; f++) {
            if (r) put(r + f * g.S, n, Cvt<TS>::st(v[f]));
            acc += (double)v[f] * v[f];
        }
    }
    if (part) {
        for (int o = 32; o > 0; o >>= 1) acc += __shfl_down(acc, o, 64);
        if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = acc;
        __syncthreads();
        if (threadIdx.x == 0) part[blockIdx.x] = sh[0] + sh[1] + sh[2] + sh[3];
    }
}

// ----------------------------------------------------------- prolongation

// xf += P ec on the free DOFs (pressure correction scaled by 1/2).  A lane takes the
// two fine nodes over one coarse entry of the fastest axis, whose coarse values they
// share; V2: rows start on even entries, and the pair moves in one access per field.
template <typename T> struct alignas(2 * sizeof(T)) Two {
    T v[2];
};
template <typename TS, int DIM, bool V2>
__global__ void __launch_bounds__(256) k_prolong(Lvl gf, Lvl gc, const uint8_t *__restrict__ flf,
                                                 const TS *__restrict__ ec, TS *__restrict__ xf)
{
    typedef typename Cvt<TS>::C C;
    const unsigned m = (unsigned)(DIM == 3 ? gc.nz : gc.ny) + 1u;  // coarse entries of a row
    const unsigned t = blockIdx.x * blockDim.x + threadIdx.x;
    const unsigned row = t / m, e = t - row * m;                    // fine row: i (2D) or i, j
    if (row >= (unsigned)(DIM == 3 ? gf.Px * gf.Py : gf.Px)) return;
    const unsigned i = DIM == 3 ? row / (unsigned)gf.Py : row, j = DIM == 3 ? row - i * (unsigned)gf.Py : 2u * e;
    const unsigned rowlen = (unsigned)(DIM == 3 ? gf.nz : gf.ny) + 1u, pitch = (unsigned)(DIM == 3 ? gf.Pz : gf.Py);
    const unsigned q = row * pitch + 2u * e;
    const unsigned qc = DIM == 3 ? ((i >> 1) * (unsigned)gc.Py + (j >> 1)) * (unsigned)gc.Pz + e
                                 : (i >> 1) * (unsigned)gc.Py + e;
    const bool two = 2u * e + 1u < rowlen;  // the last entry of a row is alone
    const long sc[3] = {(long)gc.Py * gc.Pz, (long)gc.Pz, 1};
    constexpr int fast = DIM - 1;  // axis of the pair
    int fb[2];
    if (V2) {
        const Two<uint8_t> w = *reinterpret_cast<const Two<uint8_t> *>(flf + q);
        fb[0] = w.v[0];
        fb[1] = two ? w.v[1] : 0;
    } else {
        fb[0] = at(flf, q);
        fb[1] = two ? (int)at(flf, q + 1u) : 0;
    }
    const unsigned co[3] = {i, j, 2u * e};
#pragma unroll
    for (int f = 0; f <= DIM; f++) {
        C c0 = Cvt<TS>::ld(at(ec + f * gc.S, qc)), c1;
        if (f == 0) {
            c0 = C(0.5) * c0;
            c1 = c0;
        } else if (f - 1 == fast) {
            c1 = c0 + Cvt<TS>::ld(at(ec + f * gc.S, two ? qc + 1u : qc));
            c1 *= C(0.5);
        } else {
            const bool odd = co[f - 1] & 1u;
            const C h = Cvt<TS>::ld(at(ec + f * gc.S, odd ? qc + (unsigned)sc[f - 1] : qc));
            if (odd) {
                c0 = c0 + h;
                c0 *= C(0.5);
            }
            c1 = c0;
        }
        // loads before the flag tests: a lane waits once
        TS *xp = xf + f * gf.S;
        const bool on0 = (fb[0] >> f) & 1, on1 = (fb[1] >> f) & 1;
        if (V2) {
            Two<TS> w = *reinterpret_cast<const Two<TS> *>(xp + q);
            if (on0) w.v[0] = Cvt<TS>::st(Cvt<TS>::ld(w.v[0]) + c0);
            if (on1) w.v[1] = Cvt<TS>::st(Cvt<TS>::ld(w.v[1]) + c1);
            if (on0 || on1) *reinterpret_cast<Two<TS> *>(xp + q) = w;
        } else {
            const unsigned q1 = two ? q + 1u : q;
            const TS w0 = at(xp, q), w1 = at(xp, q1);
            if (on0) put(xp, q, Cvt<TS>::st(Cvt<TS>::ld(w0) + c0));
            if (on1) put(xp, q1, Cvt<TS>::st(Cvt<TS>::ld(w1) + c1));
        }
    }
}

// ------------------------------------------------------------ LDS tiles

// A box of NI x NJ x NK nodes (NK = 1 in 2D) of x and the flags in LDS, entries outside
// the level zero, so that the stencil needs no range test and its offsets are constants
// of the LDS instructions.
template <typename TS, int DIM, int NI, int NJ, int NK> struct Tile {
    typedef typename Cvt<TS>::C C;
    static constexpr int SI = DIM == 3 ? NJ * NK : NJ, SJ = DIM == 3 ? NK : 1, SK = DIM == 3 ? 1 : 0, N = NI * NJ * NK;
    TS x[DIM + 1][N];
    uint8_t f[N];

    // nodes from (i0, j0, k0); PROL: x + P ec instead of x; ZERO: x = 0 and not read
    template <int NT, bool ZERO, bool PROL>
    __device__ __forceinline__ void load(const Lvl &g, const uint8_t *fl, const TS *xg, const Lvl &gc, const TS *ec, int i0,
                                         int j0, int k0)
    {
        static_assert(!PROL || DIM == 2, "the prolongation is fused in 2D");
#pragma unroll 2
        for (int t = threadIdx.x; t < N; t += NT) {
            int i, j, k;
            if (DIM == 3) {
                k = k0 + t % NK;
                j = j0 + (t / NK) % NJ;
                i = i0 + t / (NK * NJ);
            } else {
                k = 0;
                j = j0 + t % NJ;
                i = i0 + t / NJ;
            }
            const bool in = i >= 0 && i <= g.nx && j >= 0 && j <= g.ny && (DIM == 2 || (k >= 0 && k <= g.nz));
            const unsigned q = in ? ((unsigned)i * (unsigned)g.Py + (unsigned)j) * (unsigned)g.Pz + (unsigned)k : 0u;
            const int fb = in ? (int)at(fl, q) : 0;
            f[t] = (uint8_t)fb;
            if (ZERO) {
#pragma unroll
                for (int c = 0; c <= DIM; c++) x[c][t] = Cvt<TS>::st(C(0));
                continue;
            }
            TS v[DIM + 1];
#pragma unroll
            for (int c = 0; c <= DIM; c++) v[c] = at(xg + c * g.S, q);
            if constexpr (PROL) {  // as k_prolong
                const unsigned qc = in ? (unsigned)(i >> 1) * (unsigned)gc.Py + (unsigned)(j >> 1) : 0u;
#pragma unroll
                for (int c = 0; c <= 2; c++) {
                    C e = Cvt<TS>::ld(at(ec + c * gc.S, qc));
                    if (c == 0) {
                        e = C(0.5) * e;
                    } else {
                        const bool odd = (c == 1 ? i : j) & 1;
                        const C h = Cvt<TS>::ld(at(ec + c * gc.S, odd && in ? qc + (c == 1 ? (unsigned)gc.Py : 1u) : qc));
                        if (odd) {
                            e = e + h;
                            e *= C(0.5);
                        }
                    }
                    if ((fb >> c) & 1) v[c] = Cvt<TS>::st(Cvt<TS>::ld(v[c]) + e);
                }
            }
#pragma unroll
            for (int c = 0; c <= DIM; c++) x[c][t] = in ? v[c] : Cvt<TS>::st(C(0));
        }
    }
};

// --------------------------------------------------------- sweeps in 2D

// NPASS colour passes (first colour col0) of a 2D level in one launch: a workgroup holds
// a tile of 16 x 16 cells and a ring of 2 (NPASS - 1) cells around it in LDS and updates
// it in place, the ring losing two cells a side per pass, so no workgroup waits for
// another; the passes on the ring are done by every tile that needs them.  A lane keeps
// its pair of cells (one of each colour) and their right-hand sides and penalties in
// registers for all passes.  ZERO: x starts at zero; PROL: at xin + P ec (the
// prolongated correction).
//
// The four passes and the prolongation after the coarse correction take 9-12 us (64^2 to
// 256^2, FP32 / FP64) against five launches of 3.5-5.7 us; a whole FP64 solve 128^2 1.84 ->
// 1.54 ms, 512^2 3.08 -> 2.63, 1024^2 7.23 -> 6.60, so every 2D level takes this way.  In
// 3D the ring of one sweep is six times a tile of the same memory: measured as two
// passes per launch, 32^3 FP64 solves 2.03 -> 2.02 ms, 64^3 and 128^3 slower.
template <int NPASS> struct SwTile {
    static constexpr int H = 2 * (NPASS - 1), TI = 16, TJ = 16;
    static constexpr int RI = TI + 2 * H, RJ = TJ + 2 * H;                     // cells of the first pass
    static constexpr int NP = RI * RJ / 2, NT = (NP + 63) / 64 * 64;           // a lane per pair of them
    static constexpr int NI = RI + 3, NJ = RJ + 3;                             // nodes: one below, two above
};

// the pair's right-hand sides and penalties: x faces [high][cell], y faces low to high
template <typename C> struct PairOps {
    C p[2], bx[2][2], ax[2][2], by[3], ay[3];
};
template <typename TS, typename T, bool M> struct PairAcc {
    typedef typename Cvt<TS>::C C;
    static constexpr bool MASK = M;
    const T &t;
    const PairOps<C> &o;
    int q;
    bool par;  // the odd cell of the pair
    __device__ __forceinline__ int F(int di, int dj, int) const { return t.f[q + di * T::SI + dj * T::SJ]; }
    __device__ __forceinline__ C X(int f, int di, int dj, int) const { return Cvt<TS>::ld(t.x[f][q + di * T::SI + dj * T::SJ]); }
    // by value: a conditional between two members would be an address, and keep the
    // operands out of registers
    __device__ __forceinline__ C sel(C even, C odd) const { return par ? odd : even; }
    __device__ __forceinline__ C B(int f, int di, int dj, int) const
    { return f == 0 ? sel(o.p[0], o.p[1]) : (f == 1 ? sel(o.bx[di][0], o.bx[di][1]) : sel(o.by[dj], o.by[1 + dj])); }
    __device__ __forceinline__ C AL(int d, int di, int dj, int) const
    { return d == 0 ? sel(o.ax[di][0], o.ax[di][1]) : sel(o.ay[dj], o.ay[1 + dj]); }
};

template <typename TS, int NPASS, bool ZERO, bool PROL, bool MASK>
__global__ void __launch_bounds__(SwTile<NPASS>::NT) k_sweeps(Lvl g, Lvl gc, const uint8_t *__restrict__ fl,
                                                              const TS *__restrict__ al, const TS *__restrict__ b,
                                                              const TS *__restrict__ xin, const TS *__restrict__ ec,
                                                              TS *__restrict__ xout, int col0, float omega)
{
    typedef typename Cvt<TS>::C C;
    typedef SwTile<NPASS> W;
    typedef Tile<TS, 2, W::NI, W::NJ, 1> T;
    __shared__ T s;
    const int I0 = blockIdx.y * W::TI, J0 = blockIdx.x * W::TJ;
    // the lane's pair (i, j), (i, j + 1) in the region of the first pass
    const int t = threadIdx.x, rj = 2 * (t % (W::RJ / 2)), ri = t / (W::RJ / 2);
    const int i = I0 - W::H + ri, j = J0 - W::H + rj;
    const bool in = t < W::NP && i >= 0 && i < g.nx && j >= 0 && j < g.ny;
    const unsigned q = in ? (unsigned)i * (unsigned)g.Py + (unsigned)j : 0u;
    PairOps<C> o;
    if (in) {
        auto ldb = [&](int f, long off) -> C { return Cvt<TS>::ld(at(b + f * g.S + off, q)); };
        auto lda = [&](int d, long off) -> C { return Cvt<TS>::ld(at(al + d * g.S + off, q)); };
#pragma unroll
        for (int c = 0; c < 2; c++) {
            o.p[c] = ldb(0, c);
#pragma unroll
            for (int h = 0; h < 2; h++) {
                o.bx[h][c] = ldb(1, h * g.Py + c);
                o.ax[h][c] = lda(0, h * g.Py + c);
            }
        }
#pragma unroll
        for (int h = 0; h < 3; h++) {
            o.by[h] = ldb(2, h);
            o.ay[h] = lda(1, h);
        }
    }
    s.template load<W::NT, ZERO, PROL>(g, fl, xin, gc, ec, I0 - W::H - 1, J0 - W::H - 1, 0);
    __syncthreads();
    const int n0 = (ri + 1) * T::SI + rj + 1;  // LDS node of the even cell
#pragma unroll 1
    for (int p = 0; p < NPASS; p++) {
        const int ring = 2 * p;  // cells of the first region that this pass leaves out, a side
        const bool on = in && ri >= ring && ri < W::RI - ring && rj >= ring && rj < W::RJ - ring;
        const bool par = (i + j + col0 + p) & 1;  // which cell has this pass's colour
        const int n1 = n0 + (par ? 1 : 0);
        C pn, u0[3], u1[3];
        if (on) {
            const PairAcc<TS, T, MASK> a{s, o, n1, par};
            if (ZERO && p == 0) box_cell<C, 2, true>(a, omega, pn, u0, u1);
            else box_cell<C, 2, false>(a, omega, pn, u0, u1);
        }
        if (p + 1 < NPASS) {
            __syncthreads();
            if (on) {
                s.x[0][n1] = Cvt<TS>::st(pn);
                s.x[1][n1] = Cvt<TS>::st(u0[0]);
                s.x[1][n1 + T::SI] = Cvt<TS>::st(u1[0]);
                s.x[2][n1] = Cvt<TS>::st(u0[1]);
                s.x[2][n1 + 1] = Cvt<TS>::st(u1[1]);
            }
            __syncthreads();
        } else if (on) {  // the tile's own cells: their block, and what the colour does not own
            const unsigned qc = q + (par ? 1u : 0u), qo = q + (par ? 0u : 1u);
            const int no = n0 + (par ? 0 : 1), oj = j + (par ? 0 : 1);
            put(xout, qo, s.x[0][no]);
            if (i == 0) put(xout + g.S, qo, s.x[1][no]);
            if (i == g.nx - 1) put(xout + g.S + g.Py, qo, s.x[1][no + T::SI]);
            if (oj == 0) put(xout + 2 * g.S, qo, s.x[2][no]);
            if (oj == g.ny - 1) put(xout + 2 * g.S + 1, qo, s.x[2][no + 1]);
            put(xout, qc, Cvt<TS>::st(pn));
            put(xout + g.S, qc, Cvt<TS>::st(u0[0]));
            put(xout + g.S + g.Py, qc, Cvt<TS>::st(u1[0]));
            put(xout + 2 * g.S, qc, Cvt<TS>::st(u0[1]));
            put(xout + 2 * g.S + 1, qc, Cvt<TS>::st(u1[1]));
        }
    }
}

// ------------------------------------------------- residual + restriction

// Coarse right-hand side R (b - A x) in one launch: a workgroup stages x around its CI x
// CJ x CK coarse nodes in LDS, evaluates the fine residual on the (2 CI + 1) x (2 CJ + 1) x
// (2 CK + 1) nodes under them (rounded to the storage type, as a stored residual is) and
// restricts from LDS with restrict_body's sums.  The residual never reaches memory
// and one launch of each level's cycle is saved; 1.3-1.5 of the residual rows are
// evaluated twice, which on these levels is cheaper than a launch.
template <int DIM> struct RrTile {  // NT: one lane per residual node
    static constexpr int CI = DIM == 3 ? 2 : 4, CJ = DIM == 3 ? 4 : 16, CK = DIM == 3 ? 8 : 1;
    static constexpr int FI = 2 * CI + 1, FJ = 2 * CJ + 1, FK = DIM == 3 ? 2 * CK + 1 : 1, N = FI * FJ * FK;
    static constexpr int NT = (N + 63) / 64 * 64;
};
// a residual node in the tile: b and alpha of the own node from memory
template <typename TS, int DIM, typename T, bool M> struct RrAcc {
    typedef typename Cvt<TS>::C C;
    static constexpr bool MASK = M;
    const T &t;
    const TS *al;
    long S;
    int n0;
    unsigned q;
    __device__ __forceinline__ int n(int di, int dj, int dk) const { return n0 + di * T::SI + dj * T::SJ + dk * T::SK; }
    __device__ __forceinline__ int F(int di, int dj, int dk) const { return t.f[n(di, dj, dk)]; }
    __device__ __forceinline__ C X(int f, int di, int dj, int dk) const { return Cvt<TS>::ld(t.x[f][n(di, dj, dk)]); }
    __device__ __forceinline__ C AL(int d, int, int, int) const { return Cvt<TS>::ld(at(al + d * S, q)); }
};

// row f of the restriction at a free coarse DOF (else 0) from the residual r of field f
// around the fine node of the coarse node, strides sI, sJ, sK: the sums of restrict_body
// in its order (along the face normal, then the two axes across in (i, j, k) order)
template <typename TS, int DIM>
__device__ __forceinline__ typename Cvt<TS>::C restrict_from(const TS *r, int f, int sI, int sJ, int sK, bool free)
{
    typedef typename Cvt<TS>::C C;
    if (!free) return C(0);
    C s = C(0);
    if (f == 0) {
        for (int a = 0; a < 2; a++)
            for (int b = 0; b < 2; b++)
                for (int c = 0; c < (DIM == 3 ? 2 : 1); c++) s += Cvt<TS>::ld(r[a * sI + b * sJ + c * sK]);
        return s * ((DIM == 3) ? C(0.25) : C(0.5));
    }
    const int so = f == 1 ? sI : (f == 2 ? sJ : sK), su = f == 1 ? sJ : sI, sv = f == 3 ? sJ : sK;
    for (int on = -1; on <= 1; on++) {
        const C w = (on == 0) ? C(1) : C(0.5);
        for (int a = 0; a < 2; a++)
            for (int b = 0; b < (DIM == 3 ? 2 : 1); b++) s += w * Cvt<TS>::ld(r[on * so + a * su + b * sv]);
    }
    return s * ((DIM == 3) ? C(0.5) : C(1.0));
}

template <typename TS, int DIM, bool MASK>
__global__ void __launch_bounds__(RrTile<DIM>::NT) k_resid_restrict(Lvl gf, Lvl gc, const uint8_t *__restrict__ flf,
                                                          const TS *__restrict__ al, const TS *__restrict__ b,
                                                          const TS *__restrict__ x, const uint8_t *__restrict__ flc,
                                                          TS *__restrict__ bc)
{
    typedef typename Cvt<TS>::C C;
    typedef RrTile<DIM> T;
    typedef Tile<TS, DIM, T::FI + 2, T::FJ + 2, DIM == 3 ? T::FK + 2 : 1> X;
    __shared__ X xt;
    __shared__ TS sr[DIM + 1][T::N];
    const int K0 = blockIdx.x * T::CK, J0 = blockIdx.y * T::CJ, I0 = blockIdx.z * T::CI;
    const int t0 = threadIdx.x;
    const int fk = t0 % T::FK, fj = (t0 / T::FK) % T::FJ, fi = t0 / (T::FK * T::FJ);
    const int i = 2 * I0 - 1 + fi, j = 2 * J0 - 1 + fj, k = DIM == 3 ? 2 * K0 - 1 + fk : 0;
    const bool in = t0 < T::N && i >= 0 && j >= 0 && k >= 0 && i <= gf.nx && j <= gf.ny && (DIM == 2 || k <= gf.nz);
    const unsigned q = in ? ((unsigned)i * (unsigned)gf.Py + (unsigned)j) * (unsigned)gf.Pz + (unsigned)k : 0u;
    C v[4];
#pragma unroll
    for (int f = 0; f <= DIM; f++) v[f] = Cvt<TS>::ld(at(b + f * gf.S, q));
    xt.template load<T::NT, false, false>(gf, flf, x, gc, (const TS *)nullptr, 2 * I0 - 2, 2 * J0 - 2,
                                          DIM == 3 ? 2 * K0 - 2 : 0);
    __syncthreads();
    if (t0 < T::N) {
        const RrAcc<TS, DIM, X, MASK> a{xt, al, gf.S, (fi + 1) * X::SI + (fj + 1) * X::SJ + (DIM == 3 ? fk + 1 : 0), q};
        const BoxSten<C, DIM, RrAcc<TS, DIM, X, MASK>> s{a};
        v[0] -= s.cell();
        v[1] -= s.template face<0>(0, 0, 0);
        v[2] -= s.template face<1>(0, 0, 0);
        if (DIM == 3) v[3] -= s.template face<2>(0, 0, 0);
#pragma unroll
        for (int f = 0; f <= DIM; f++) sr[f][t0] = Cvt<TS>::st(in ? v[f] : C(0));
    }
    __syncthreads();
    constexpr int NC = T::CI * T::CJ * T::CK;
    for (int t = threadIdx.x; t < NC * (DIM + 1); t += T::NT) {
        const int f = t / NC, n = t % NC;
        const int dK = n % T::CK, dJ = (n / T::CK) % T::CJ, dI = n / (T::CK * T::CJ);
        const int I = I0 + dI, J = J0 + dJ, K = K0 + dK;
        if (I > gc.nx || J > gc.ny || (DIM == 3 && K > gc.nz)) continue;
        const unsigned qc = ((unsigned)I * (unsigned)gc.Py + (unsigned)J) * (unsigned)gc.Pz + (unsigned)K;
        const C s = restrict_from<TS, DIM>(
            &sr[f][((2 * dI + 1) * T::FJ + (2 * dJ + 1)) * T::FK + (DIM == 3 ? 2 * dK + 1 : 0)], f, T::FJ * T::FK, T::FK,
            DIM == 3 ? 1 : 0, (at(flc, qc) >> f) & 1);
        put(bc + f * gc.S, qc, Cvt<TS>::st(s));
    }
}

// ------------------------------------------------ fused coarsest levels

namespace {

// One level of the fused cycle in LDS, side N known to the compiler.  Every field is a
// box of (N + 2)^DIM nodes, indices -1 .. N per axis: the zero entries at -1 stand for
// everything outside the level (the entry after N along an axis is the -1 of the next
// row or plane; after the last plane of u_x comes u_y's, after the flags a spare plane).
template <typename TS, int DIM, int N> struct TLvl {
    static constexpr int P = N + 2, SK = DIM == 3 ? 1 : 0, SJ = DIM == 3 ? P : 1, SI = SJ * P;
    static constexpr int NODES = SI * P, NF = DIM + 1;
    static constexpr int VEC = NF * NODES;
    static constexpr bool LAST = N == 2;          // coarsest: only b and x are kept
    TS x[VEC], b[VEC];
    TS al[LAST ? 1 : DIM * NODES], r[LAST ? 1 : VEC];
    uint8_t fl[(NODES + SI + 15) / 16 * 16];
    __device__ static constexpr int id(int i, int j, int k) { return (i + 1) * SI + (j + 1) * SJ + (DIM == 3 ? (k + 1) * SK : 0); }
};

template <typename TS, int DIM, int N, bool M> struct LdsAcc {
    typedef typename Cvt<TS>::C C;
    static constexpr bool MASK = M;
    typedef TLvl<TS, DIM, N> L;
    const L &l;
    int q;
    __device__ __forceinline__ int o(int di, int dj, int dk) const { return q + di * L::SI + dj * L::SJ + dk * L::SK; }
    __device__ __forceinline__ int F(int di, int dj, int dk) const { return l.fl[o(di, dj, dk)]; }
    __device__ __forceinline__ C X(int f, int di, int dj, int dk) const { return Cvt<TS>::ld(l.x[f * L::NODES + o(di, dj, dk)]); }
    __device__ __forceinline__ C B(int f, int di, int dj, int dk) const { return Cvt<TS>::ld(l.b[f * L::NODES + o(di, dj, dk)]); }
    __device__ __forceinline__ C AL(int d, int di, int dj, int dk) const { return Cvt<TS>::ld(l.al[d * L::NODES + o(di, dj, dk)]); }
};

// What a colour cell of the lane keeps in registers over the level's passes of a cycle: its
// right-hand side, penalties and the flags of its node and the neighbours along the axes,
// half of what a pass reads from LDS and, with BF16 storage, converts (the cycle from 32^2
// 50 -> 36 us BF16, 31 -> 29 FP32; from 8^3 35 -> 27 and 24 -> 23).  Not in FP64, where
// they spill: 38 -> 47 us from 32^2, and read again on the way up 38 -> 38.
template <typename TS, int DIM> struct TailCell {
    typename Cvt<TS>::C b[1 + 2 * DIM], al[2 * DIM];
    int fl, q;
};
template <typename TS> constexpr bool tail_keep() { return sizeof(typename Cvt<TS>::C) == 4; }
template <typename TS, int DIM, int N, bool M> struct TailAcc {
    typedef typename Cvt<TS>::C C;
    static constexpr bool MASK = M, KEEP = tail_keep<TS>();
    LdsAcc<TS, DIM, N, M> a;
    TailCell<TS, DIM> c;
    __device__ __forceinline__ int F(int di, int dj, int dk) const
    {
        const int s = di + dj + dk, ax = di ? 0 : (dj ? 1 : 2);
        if (!KEEP || (di != 0) + (dj != 0) + (dk != 0) > 1 || s > 1 || s < -1) return a.F(di, dj, dk);
        return (c.fl >> (s == 0 ? 0 : 4 * (1 + 2 * ax + (s > 0)))) & 15;
    }
    __device__ __forceinline__ C X(int f, int di, int dj, int dk) const { return a.X(f, di, dj, dk); }
    __device__ __forceinline__ C B(int f, int di, int dj, int dk) const
    { return KEEP ? c.b[di + dj + dk ? DIM + f : f] : a.B(f, di, dj, dk); }
    __device__ __forceinline__ C AL(int d, int di, int dj, int dk) const
    { return KEEP ? c.al[di + dj + dk ? DIM + d : d] : a.AL(d, di, dj, dk); }
};

constexpr int TAIL_NT = 512;  // 256 registers a lane: the FP64 block solve fits them

// the node t of the (N + 1)^DIM nodes of a level
template <int DIM, int N> __device__ __forceinline__ void node_of(int t, int &i, int &j, int &k)
{
    if (DIM == 3) {
        k = t % (N + 1);
        j = (t / (N + 1)) % (N + 1);
        i = t / ((N + 1) * (N + 1));
    } else {
        k = 0;
        j = t % (N + 1);
        i = t / (N + 1);
    }
}
template <int DIM, int N> constexpr int n_nodes() { return (N + 1) * (N + 1) * (DIM == 3 ? N + 1 : 1); }

// the lane's cell of a colour (the first half of the level's cells, one per lane)
template <typename TS, int DIM, int N, bool MASK>
__device__ __forceinline__ TailCell<TS, DIM> tail_cell(const TLvl<TS, DIM, N> &l, int color)
{
    typedef TLvl<TS, DIM, N> L;
    constexpr int NP = (DIM == 3 ? N * N * N : N * N) / 2, H = N / 2;
    static_assert(NP <= TAIL_NT, "one colour cell per lane");
    const int t = (int)threadIdx.x < NP ? (int)threadIdx.x : 0;
    int i, j, k;
    const int pr = 2 * (t % H);
    if (DIM == 3) {
        j = (t / H) % N;
        i = t / (H * N);
        k = pr + ((i + j + color) & 1);
    } else {
        i = t / H;
        j = pr + ((i + color) & 1);
        k = 0;
    }
    TailCell<TS, DIM> c;
    c.q = L::id(i, j, k);
    if (!tail_keep<TS>()) return c;
    const LdsAcc<TS, DIM, N, MASK> a{l, c.q};
    c.fl = a.F(0, 0, 0) & 15;
    c.b[0] = a.B(0, 0, 0, 0);
#pragma unroll
    for (int d = 0; d < DIM; d++) {
        const int di = d == 0, dj = d == 1, dk = d == 2;
        c.fl |= (a.F(-di, -dj, -dk) & 15) << (4 * (1 + 2 * d)) | (a.F(di, dj, dk) & 15) << (4 * (2 + 2 * d));
        c.b[1 + d] = a.B(1 + d, 0, 0, 0);
        c.b[1 + DIM + d] = a.B(1 + d, di, dj, dk);
        c.al[d] = a.AL(d, 0, 0, 0);
        c.al[DIM + d] = a.AL(d, di, dj, dk);
    }
    return c;
}

// one colour pass in place: every lane reads what it needs, then every lane writes (the
// first pass of the way down reads the zeros the launch starts with)
template <typename TS, int DIM, int N, bool MASK>
__device__ __forceinline__ void tail_color(TLvl<TS, DIM, N> &l, const TailCell<TS, DIM> &c, float omega)
{
    typedef typename Cvt<TS>::C C;
    typedef TLvl<TS, DIM, N> L;
    constexpr int NP = (DIM == 3 ? N * N * N : N * N) / 2;
    const int t = threadIdx.x, q = c.q;
    C pn, u0[3], u1[3];
    if (t < NP) {
        const TailAcc<TS, DIM, N, MASK> a{{l, q}, c};
        box_cell<C, DIM, false>(a, omega, pn, u0, u1);
    }
    __syncthreads();
    if (t < NP) {
        l.x[q] = Cvt<TS>::st(pn);
        const int st[3] = {L::SI, L::SJ, L::SK};
#pragma unroll
        for (int d = 0; d < DIM; d++) {
            l.x[(1 + d) * L::NODES + q] = Cvt<TS>::st(u0[d]);
            l.x[(1 + d) * L::NODES + q + st[d]] = Cvt<TS>::st(u1[d]);
        }
    }
    __syncthreads();
}

template <typename TS, int DIM, int N, bool MASK>
__device__ __forceinline__ void tail_smooth(TLvl<TS, DIM, N> &l, const TailCell<TS, DIM> &c0, const TailCell<TS, DIM> &c1,
                                            int nu, int first, float omega)
{
#pragma unroll 1
    for (int s = 0; s < 2 * nu; s++) {
        const bool odd = first ^ (s & 1);
        TailCell<TS, DIM> c;
        c.q = odd ? c1.q : c0.q;
        if (tail_keep<TS>()) {
            c.fl = odd ? c1.fl : c0.fl;
#pragma unroll
            for (int v = 0; v < 1 + 2 * DIM; v++) c.b[v] = odd ? c1.b[v] : c0.b[v];
#pragma unroll
            for (int v = 0; v < 2 * DIM; v++) c.al[v] = odd ? c1.al[v] : c0.al[v];
        }
        tail_color<TS, DIM, N, MASK>(l, c, omega);
    }
}

// r = b - A x on the nodes of the level
template <typename TS, int DIM, int N, bool MASK>
__device__ __forceinline__ void tail_residual(TLvl<TS, DIM, N> &l)
{
    typedef typename Cvt<TS>::C C;
    typedef TLvl<TS, DIM, N> L;
    for (int t = threadIdx.x; t < n_nodes<DIM, N>(); t += TAIL_NT) {
        int i, j, k;
        node_of<DIM, N>(t, i, j, k);
        const LdsAcc<TS, DIM, N, MASK> a{l, L::id(i, j, k)};
        const BoxSten<C, DIM, LdsAcc<TS, DIM, N, MASK>> s{a};
        l.r[a.q] = Cvt<TS>::st(a.B(0, 0, 0, 0) - s.cell());
        l.r[L::NODES + a.q] = Cvt<TS>::st(a.B(1, 0, 0, 0) - s.template face<0>(0, 0, 0));
        l.r[2 * L::NODES + a.q] = Cvt<TS>::st(a.B(2, 0, 0, 0) - s.template face<1>(0, 0, 0));
        if (DIM == 3) l.r[3 * L::NODES + a.q] = Cvt<TS>::st(a.B(3, 0, 0, 0) - s.template face<2>(0, 0, 0));
    }
    __syncthreads();
}

// c.b = R l.r: one (field, coarse node) per lane
template <typename TS, int DIM, int N>
__device__ __forceinline__ void tail_restrict(const TLvl<TS, DIM, N> &l, TLvl<TS, DIM, N / 2> &c)
{
    typedef typename Cvt<TS>::C C;
    typedef TLvl<TS, DIM, N> L;
    typedef TLvl<TS, DIM, N / 2> K_;
    constexpr int NN = n_nodes<DIM, N / 2>();
    for (int t = threadIdx.x; t < NN * (DIM + 1); t += TAIL_NT) {
        const int f = t / NN;
        int I, J, K;
        node_of<DIM, N / 2>(t % NN, I, J, K);
        const int qc = K_::id(I, J, K), q = L::id(2 * I, 2 * J, 2 * K);
        const C s = restrict_from<TS, DIM>(l.r + f * L::NODES + q, f, L::SI, L::SJ, L::SK, (c.fl[qc] >> f) & 1);
        c.b[f * K_::NODES + qc] = Cvt<TS>::st(s);
    }
    __syncthreads();
}

// l.x += P c.x on the free DOFs
template <typename TS, int DIM, int N>
__device__ __forceinline__ void tail_prolong(TLvl<TS, DIM, N> &l, const TLvl<TS, DIM, N / 2> &c)
{
    typedef typename Cvt<TS>::C C;
    typedef TLvl<TS, DIM, N> L;
    typedef TLvl<TS, DIM, N / 2> K_;
    for (int t = threadIdx.x; t < n_nodes<DIM, N>(); t += TAIL_NT) {
        int co[3];
        node_of<DIM, N>(t, co[0], co[1], co[2]);
        const int q = L::id(co[0], co[1], co[2]), qc = K_::id(co[0] >> 1, co[1] >> 1, co[2] >> 1);
        const int fb = l.fl[q], st[3] = {K_::SI, K_::SJ, K_::SK};
        if (fb & 1) l.x[q] = Cvt<TS>::st(Cvt<TS>::ld(l.x[q]) + C(0.5) * Cvt<TS>::ld(c.x[qc]));
#pragma unroll
        for (int d = 0; d < DIM; d++) {
            if (!((fb >> (1 + d)) & 1)) continue;
            const TS *e0 = c.x + (1 + d) * K_::NODES + qc;
            C e = Cvt<TS>::ld(e0[0]);
            if (co[d] & 1) {
                e += Cvt<TS>::ld(e0[st[d]]);
                e *= C(0.5);
            }
            TS &v = l.x[(1 + d) * L::NODES + q];
            v = Cvt<TS>::st(Cvt<TS>::ld(v) + e);
        }
    }
    __syncthreads();
}

// level data from the node layout of device memory (levels below 64 a side: pitch N + 1)
template <typename TS, int DIM, int N>
__device__ __forceinline__ void tail_load(TLvl<TS, DIM, N> &l, const uint8_t *fl, const TS *al, const TS *b)
{
    typedef TLvl<TS, DIM, N> L;
    constexpr int NN = n_nodes<DIM, N>();
    for (int t = threadIdx.x; t < NN; t += TAIL_NT) {
        int i, j, k;
        node_of<DIM, N>(t, i, j, k);
        const int q = L::id(i, j, k);
        l.fl[q] = fl[t];
        if constexpr (!L::LAST)
            for (int d = 0; d < DIM; d++) l.al[d * L::NODES + q] = al[d * NN + t];
        if (b)
            for (int f = 0; f <= DIM; f++) l.b[f * L::NODES + q] = b[f * NN + t];
    }
}

template <typename TS, int DIM, int N> struct TailPool {
    TLvl<TS, DIM, N> l;
    TailPool<TS, DIM, N / 2> next;
};
template <typename TS, int DIM> struct TailPool<TS, DIM, 2> {
    TLvl<TS, DIM, 2> l;
};

template <typename TS, int DIM, int N, int LEV>
__device__ __forceinline__ void tail_load_all(TailPool<TS, DIM, N> &p, const TailArgs<TS> &a, const TS *b)
{
    tail_load<TS, DIM, N>(p.l, a.fl[LEV], a.al[LEV], b);
    if constexpr (N > 2) tail_load_all<TS, DIM, N / 2, LEV + 1>(p.next, a, nullptr);
}

// DOFs of the coarsest level (2 cells a side) in the compact list's order
template <int DIM> struct TailDofs {
    static constexpr int PL = DIM == 3 ? 2 : 1;             // nodes along k
    static constexpr int NCELL = 4 * PL, NFACE = 6 * PL;    // per direction (i and j: 3 x 2 x PL; k: 2 x 2 x 3)
    static constexpr int ND = NCELL + DIM * NFACE;
    static constexpr int LPR = 8, NCOL = (ND + LPR - 1) / LPR;  // lanes per row, columns per lane
};
// position of the compact DOF c in the coarsest level's LDS box
template <typename TS, int DIM> __device__ __forceinline__ int tail_dof(int c)
{
    typedef TLvl<TS, DIM, 2> L;
    typedef TailDofs<DIM> D;
    const int f = c < D::NCELL ? 0 : 1 + (c - D::NCELL) / D::NFACE;
    const int m = c < D::NCELL ? c : (c - D::NCELL) % D::NFACE;
    const int nk = DIM == 3 ? 2 + (f == 3) : 1, nj = 2 + (f == 2);
    return f * L::NODES + L::id(m / (nk * nj), (m / nk) % nj, m % nk);
}

// rows of the coarsest inverse held by a lane: LPR lanes per row, columns lane, lane + LPR, ..
template <typename TS, int DIM>
__device__ __forceinline__ void tail_coarse(TLvl<TS, DIM, 2> &l, const double *mrow, const int *mcol, int row, int nd)
{
    typedef typename Cvt<TS>::C C;
    typedef TailDofs<DIM> D;
    double s = 0.0;
#pragma unroll
    for (int c = 0; c < D::NCOL; c++) s += mrow[c] * (double)Cvt<TS>::ld(l.b[mcol[c]]);
#pragma unroll
    for (int o = D::LPR / 2; o > 0; o >>= 1) s += __shfl_xor(s, o, D::LPR);
    if (row < nd && (threadIdx.x & (D::LPR - 1)) == 0) l.x[tail_dof<TS, DIM>(row)] = Cvt<TS>::st((C)s);
    __syncthreads();
}

template <typename TS, int DIM, int N, bool MASK>
__device__ __forceinline__ void tail_cycle(TailPool<TS, DIM, N> &p, int nu_pre, int nu_post, float om,
                                           const double *mrow, const int *mcol, int row, int nd)
{
    if constexpr (N == 2) {
        tail_coarse<TS, DIM>(p.l, mrow, mcol, row, nd);
    } else {
        // way down, then way up: one loop, so that the passes of a level are compiled once
        // (the launch runs on one CU, and fetching its instructions is a good part of it)
        const TailCell<TS, DIM> c0 = tail_cell<TS, DIM, N, MASK>(p.l, 0), c1 = tail_cell<TS, DIM, N, MASK>(p.l, 1);
#pragma unroll 1
        for (int up = 0; up < 2; up++) {
            if (up) tail_prolong<TS, DIM, N>(p.l, p.next.l);
            tail_smooth<TS, DIM, N, MASK>(p.l, c0, c1, up ? nu_post : nu_pre, up, om);
            if (!up) {
                tail_residual<TS, DIM, N, MASK>(p.l);
                tail_restrict<TS, DIM, N>(p.l, p.next.l);
                tail_cycle<TS, DIM, N / 2, false>(p.next, nu_pre, nu_post, om, mrow, mcol, row, nd);
            }
        }
    }
}

}  // namespace

// The V-cycle from a level of N cells a side (8 in 3D; 32, or the grid itself, in 2D)
// down to the coarsest one and back in one workgroup, every buffer in LDS.  x is
// updated in place (a pass holds its results in registers over a barrier), so a level
// needs x, b, alpha and r only and a 32^2 level fits in FP64; sides, pitches and loop
// counts are compile-time constants, and the coarsest inverse is read into registers
// while the levels are staged.  Per cycle, first level 8^3: 28 us FP64, 23 us FP32
// (81 us both with 64-bit index arithmetic, run-time sides and the rows of a cell
// evaluated one by one); from 32^2: 38 / 29 us (65 us from 16^2, and ten launches of
// 3-7 us for the 32^2 level).  One workgroup is a chain of ~20 passes of ~1 us each.
template <typename TS, int DIM, int N, bool MASK>
__global__ void __launch_bounds__(TAIL_NT) k_tail(TailArgs<TS> a, const TS *__restrict__ b0, TS *__restrict__ x0)
{
    typedef TailPool<TS, DIM, N> Pool;
    typedef TailDofs<DIM> D;
    static_assert(sizeof(Pool) <= 160 * 1024, "the levels of the fused cycle fit in LDS");
    static_assert(D::ND * D::LPR <= TAIL_NT, "a row of the coarsest inverse per group of lanes");
    __shared__ __align__(16) unsigned char mem[sizeof(Pool) / 16 * 16 + 16];
    Pool &p = *reinterpret_cast<Pool *>(mem);
    const int nd = a.nd;
    double mrow[D::NCOL];
    int mcol[D::NCOL];
    const int row = threadIdx.x / D::LPR;
#pragma unroll
    for (int c = 0; c < D::NCOL; c++) {
        const int col = (int)(threadIdx.x & (D::LPR - 1)) + c * D::LPR;
        const bool on = row < nd && col < nd;
        mrow[c] = on ? a.minv[(long)row * nd + col] : 0.0;
        mcol[c] = on ? tail_dof<TS, DIM>(col) : 0;
    }
    for (int q = threadIdx.x; q < (int)(sizeof(mem) / 16); q += TAIL_NT)
        reinterpret_cast<uint4 *>(mem)[q] = make_uint4(0u, 0u, 0u, 0u);
    __syncthreads();
    tail_load_all<TS, DIM, N, 0>(p, a, b0);
    __syncthreads();
    tail_cycle<TS, DIM, N, MASK>(p, a.nu_pre, a.nu_post, a.omega, mrow, mcol, row, nd);
    constexpr int NN = n_nodes<DIM, N>();
    for (int t = threadIdx.x; t < NN; t += TAIL_NT) {
        int i, j, k;
        node_of<DIM, N>(t, i, j, k);
        const int q = TLvl<TS, DIM, N>::id(i, j, k);
        for (int f = 0; f <= DIM; f++) x0[f * NN + t] = p.l.x[f * TLvl<TS, DIM, N>::NODES + q];
    }
}

// ============================================================== launchers

static int lg2(int n) { return __builtin_ctz((unsigned)n); }

template <typename TS>
void launch_box(const Lvl &g, const uint8_t *fl, const TS *al, const TS *b, const TS *xin, TS *xout, int color,
                float omega, bool zero, bool inner, bool fine, hipStream_t s)
{
    const int lg = lg2(g.nx);
    const unsigned np = 1u << (g.dim * lg - 1);
    // one wave per workgroup on the smallest levels, so that every wave has a CU
    const unsigned bs = np <= (1u << 16) ? 64 : 256;
    const dim3 gr((np + bs - 1) / bs), bl(bs);
#define ST_BOX(D, Z, M, F) \
    hipLaunchKernelGGL((k_box<TS, D, Z, M, F>), gr, bl, 0, s, g, lg, fl, al, b, xin, xout, color, omega)
    if (g.dim == 3) {
        if (zero) ST_BOX(3, true, false, false);  // reads no x
        else if (fine) ST_BOX(3, false, true, true);
        else if (inner) ST_BOX(3, false, false, false);
        else ST_BOX(3, false, true, false);
    } else {  // a single pass in 2D: st_mg_smooth (a cycle's passes run in k_sweeps)
        ST_BOX(2, false, true, false);
    }
#undef ST_BOX
}

template <typename TS, int NPASS, bool ZERO, bool PROL>
static void sweeps_go(const Lvl &g, const Lvl &gc, const uint8_t *fl, const TS *al, const TS *b, const TS *xin,
                      const TS *ec, TS *xout, int col0, float omega, bool inner, hipStream_t s)
{
    typedef SwTile<NPASS> W;
    const dim3 gr((unsigned)((g.ny + W::TJ - 1) / W::TJ), (unsigned)((g.nx + W::TI - 1) / W::TI)), bl(W::NT);
    if (inner)
        hipLaunchKernelGGL((k_sweeps<TS, NPASS, ZERO, PROL, false>), gr, bl, 0, s, g, gc, fl, al, b, xin, ec, xout, col0,
                           omega);
    else
        hipLaunchKernelGGL((k_sweeps<TS, NPASS, ZERO, PROL, true>), gr, bl, 0, s, g, gc, fl, al, b, xin, ec, xout, col0,
                           omega);
}

template <typename TS>
void launch_sweeps(const Lvl &g, const Lvl &gc, const uint8_t *fl, const TS *al, const TS *b, const TS *xin, const TS *ec,
                   TS *xout, int nsweep, int col0, float omega, bool zero, bool inner, hipStream_t s)
{
#define ST_SW(NP, Z, P) sweeps_go<TS, NP, Z, P>(g, gc, fl, al, b, xin, ec, xout, col0, omega, inner, s)
    if (nsweep == 1) {
        if (zero) ST_SW(2, true, false);
        else if (ec) ST_SW(2, false, true);
        else ST_SW(2, false, false);
    } else {
        if (zero) ST_SW(4, true, false);
        else if (ec) ST_SW(4, false, true);
        else ST_SW(4, false, false);
    }
#undef ST_SW
}

template <typename TS>
void launch_resid_restrict(const Lvl &gf, const Lvl &gc, const uint8_t *flf, const TS *al, const TS *b, const TS *x,
                           const uint8_t *flc, TS *bc, bool inner, hipStream_t s)
{
    auto up = [](int n, int c) { return (unsigned)((n + c) / c); };  // n + 1 coarse nodes in tiles of c
    const dim3 g3(up(gc.nz, RrTile<3>::CK), up(gc.ny, RrTile<3>::CJ), up(gc.nx, RrTile<3>::CI));
    const dim3 g2(1, up(gc.ny, RrTile<2>::CJ), up(gc.nx, RrTile<2>::CI));
#define ST_RR(D, M, GR) \
    hipLaunchKernelGGL((k_resid_restrict<TS, D, M>), GR, dim3(RrTile<D>::NT), 0, s, gf, gc, flf, al, b, x, flc, bc)
    if (gf.dim == 3) {
        if (inner) ST_RR(3, false, g3);
        else ST_RR(3, true, g3);
    } else {
        if (inner) ST_RR(2, false, g2);
        else ST_RR(2, true, g2);
    }
#undef ST_RR
}

template <typename TS>
void launch_node_apply(const Lvl &g, const uint8_t *fl, const TS *al, const TS *x, TS *y, hipStream_t s)
{
    const dim3 gr((unsigned)((g.S + 255) / 256)), bl(256);
    if (g.dim == 3) hipLaunchKernelGGL((k_apply<TS, 3>), gr, bl, 0, s, g, fl, al, x, y);
    else hipLaunchKernelGGL((k_apply<TS, 2>), gr, bl, 0, s, g, fl, al, x, y);
}
template <typename TS>
void launch_node_residual(const Lvl &g, const uint8_t *fl, const TS *al, const TS *b, const TS *x, TS *r, double *part,
                          hipStream_t s)
{
    const dim3 gr((unsigned)((g.S + 255) / 256)), bl(256);
    if (g.dim == 3) hipLaunchKernelGGL((k_residual<TS, 3>), gr, bl, 0, s, g, fl, al, b, x, r, part);
    else hipLaunchKernelGGL((k_residual<TS, 2>), gr, bl, 0, s, g, fl, al, b, x, r, part);
}

template <typename TS>
void launch_prolong(const Lvl &gf, const Lvl &gc, const uint8_t *flf, const TS *ec, TS *xf, hipStream_t s)
{
    const long rows = gf.dim == 3 ? (long)gf.Px * gf.Py : gf.Px, m = (gf.dim == 3 ? gc.nz : gc.ny) + 1;
    const dim3 gr((unsigned)((rows * m + 255) / 256)), bl(256);
    if (gf.dim == 2) hipLaunchKernelGGL((k_prolong<TS, 2, false>), gr, bl, 0, s, gf, gc, flf, ec, xf);
    else if (gf.Pz % 2 == 0) hipLaunchKernelGGL((k_prolong<TS, 3, true>), gr, bl, 0, s, gf, gc, flf, ec, xf);
    else hipLaunchKernelGGL((k_prolong<TS, 3, false>), gr, bl, 0, s, gf, gc, flf, ec, xf);
}

template <typename TS>
void launch_vcycle_tail(const TailArgs<TS> &a, int dim, int n, const TS *b0, TS *x0, bool inner, hipStream_t s)
{
#define ST_TAIL(D, N, M) hipLaunchKernelGGL((k_tail<TS, D, N, M>), dim3(1), dim3(TAIL_NT), 0, s, a, b0, x0)
    if (dim == 3) {
        if (inner) ST_TAIL(3, 8, false);
        else ST_TAIL(3, 8, true);
    } else if (n == 32) {
        if (inner) ST_TAIL(2, 32, false);
        else ST_TAIL(2, 32, true);
    } else if (n == 16) {  // these sides start the cycle only as the grid itself
        ST_TAIL(2, 16, true);
    } else {
        ST_TAIL(2, 8, true);
    }
#undef ST_TAIL
}

#define INST_C(T)                                                                                                  \
    template void launch_box<T>(const Lvl &, const uint8_t *, const T *, const T *, const T *, T *, int, float, bool, \
                                bool, bool, hipStream_t);                                                                     \
    template void launch_resid_restrict<T>(const Lvl &, const Lvl &, const uint8_t *, const T *, const T *,       \
                                           const T *, const uint8_t *, T *, bool, hipStream_t);                   \
    template void launch_sweeps<T>(const Lvl &, const Lvl &, const uint8_t *, const T *, const T *, const T *, const T *, \
                                   T *, int, int, float, bool, bool, hipStream_t);                                \
    template void launch_node_apply<T>(const Lvl &, const uint8_t *, const T *, const T *, T *, hipStream_t);      \
    template void launch_node_residual<T>(const Lvl &, const uint8_t *, const T *, const T *, const T *, T *,     \
                                          double *, hipStream_t);                                                 \
    template void launch_prolong<T>(const Lvl &, const Lvl &, const uint8_t *, const T *, T *, hipStream_t);      \
    template void launch_vcycle_tail<T>(const TailArgs<T> &, int, int, const T *, T *, bool, hipStream_t);
INST_C(double)
INST_C(float)
INST_C(bf16)

}  // namespace st
