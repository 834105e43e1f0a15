// Operator and residual of the finest 3D levels (64 cells a side and up) without LDS.
//
// A lane takes V consecutive nodes of a row (16 bytes of a field), reads every row of
// every field it needs in one aligned access (23 of them, and single values at the row
// segment's ends), and forms each edge curl and divergence once for its nodes; the
// reuse between neighbouring rows and planes is left to L1 and L2.  The levels have no
// barrier, no staging and a wave per 64 V nodes, so a 64^3 level fills the chip where
// tiles marched through chunks of planes give it 128 workgroups.  The arithmetic is that
// of the marching kernels (st_march.hip), bit for bit.
//
// Per launch, us, against the marching kernel (LDS planes, two barriers per plane):
//                     256^3 FP64  FP32   128^3 FP64  FP32   64^3 FP64  FP32
//   y = A x           540 -> 443  262 -> 225   88 -> 66  35 -> 24   31 -> 10  24 -> 9
//   r = b - A x       627 -> 528  316 -> 245  101 -> 73  44 -> 32   36 -> 13  28 -> 10
// At 256^3 the HBM traffic is 1.79 / 2.30 GB in FP64 and 0.84 / 1.13 GB in FP32, 1.1 to 1.2
// times the least, at 3.5 to 4.4 TB/s.
// Without the masks it gains 10% in FP64 and nothing in FP32, and with fewer registers
// or other block orders nothing: the mix of 9 to 15 streams and short waves bounds it.
#include "st_box.h"
#include "st_kernels.h"

#include <type_traits>

namespace st {

namespace {
// N consecutive values at one element offset, one aligned access of a native vector
// type (an aggregate would be taken apart into one load per member)
template <typename T, int N> struct Vec {
    typedef T E;
    typedef E R __attribute__((ext_vector_type(N)));
    R v;
    __device__ __forceinline__ T get(int k) const { return v[k]; }
    __device__ __forceinline__ void set(int k, T x) { v[k] = x; }
};
template <int N> struct Vec<bf16, N> {
    typedef uint16_t R __attribute__((ext_vector_type(N)));
    R v;
    __device__ __forceinline__ bf16 get(int k) const { return bf16{v[k]}; }
    __device__ __forceinline__ void set(int k, bf16 x) { v[k] = x.v; }
};
template <int N, typename T> __device__ __forceinline__ Vec<T, N> vat(const T *p, unsigned i)
{
    Vec<T, N> r;
    r.v = *reinterpret_cast<const typename Vec<T, N>::R *>(reinterpret_cast<const char *>(p) + i * (unsigned)sizeof(T));
    return r;
}
template <int N, typename T> __device__ __forceinline__ void vput(T *p, unsigned i, const Vec<T, N> &x)
{
    // (nontemporal: x, read three times, keeps the caches: 3% at 128^3 and 256^3, 5 to 10% at 64^3)
    typedef typename Vec<T, N>::R R;
    __builtin_nontemporal_store(x.v, reinterpret_cast<R *>(reinterpret_cast<char *>(p) + i * (unsigned)sizeof(T)));
}
template <int V> struct FlagWord;
template <> struct FlagWord<2> { typedef uint16_t T; };
template <> struct FlagWord<4> { typedef uint32_t T; };

// The node kc of the lane's V consecutive nodes from offset q.  Nothing is tested for the
// edges of the level: vectors and flags have a zero plane before the first one and room
// for one after the last (st_solver.hip), so every read is in bounds; the flags outside
// are 0, which masks whatever a velocity or a cell reads below the first or past the
// last plane; and what a pressure, which is not masked, reads before the first plane,
// row or column of the level is a zero plane or an entry that is always 0 (u_z at
// i = nx before a slot of the Krylov basis, p at j = ny, the row padding).
template <typename TS, typename TX, int V> struct FineAcc {
    typedef typename Cvt<TS>::C C;
    static constexpr bool MASK = true;
    const uint8_t *fl;
    const TX *x;
    const TS *al;
    long S, sI, sJ;
    unsigned q;
    int kc;
    __device__ __forceinline__ long uni(int di, int dj) const { return di * sI + dj * sJ; }
    template <typename T> __device__ __forceinline__ T get(const T *p, int k) const
    {
        if (k >= 0 && k < V) return vat<V>(p, q).get(k);
        return at(p + k, q);
    }
    __device__ __forceinline__ int F(int di, int dj, int dk) const
    {
        const int k = kc + dk;
        const uint8_t *p = fl + uni(di, dj);
        if (k >= 0 && k < V)
            return (int)((*reinterpret_cast<const typename FlagWord<V>::T *>(p + q) >> (8 * k)) & 0xff);
        return at(p + k, q);
    }
    __device__ __forceinline__ C X(int f, int di, int dj, int dk) const { return (C)Cvt<TX>::ld(get(x + f * S + uni(di, dj), kc + dk)); }
    __device__ __forceinline__ C AL(int d, int di, int dj, int dk) const { return Cvt<TS>::ld(get(al + d * S + uni(di, dj), kc + dk)); }
};

// consecutive nodes of a lane: 16 bytes of a field (8 in BF16)
template <typename TS> constexpr int lane_nodes() { return sizeof(TS) == 8 ? 2 : 4; }
template <typename TS> static int plane_blocks(const Lvl &g) { return (int)(((long)g.Py * g.Pz / lane_nodes<TS>() + 255) / 256); }

// Block -> (plane, block of the plane): XCD x takes a run of planes and sweeps them in
// strips of sb blocks, so that the rows and planes its blocks share meet in its L2.
constexpr int STRIP = 32;  // 8 to 64 within 2% at 256^3
__device__ __forceinline__ bool strip_of(int nplane, int nb, int sb, int &i, int &blk)
{
    const int pl = (nplane + 7) >> 3;
    const int xcd = blockIdx.x & 7, r = blockIdx.x >> 3;
    const int s = r / (pl * sb), m = r - s * (pl * sb);
    i = xcd * pl + m / sb;
    blk = s * sb + m % sb;
    return i < nplane && m / sb < pl && blk < nb;
}
static unsigned strip_grid(int nplane, int nb, int sb) { return 8u * (unsigned)(((nplane + 7) >> 3) * sb * ((nb + sb - 1) / sb)); }
}  // namespace

// y = A x, or y = b - A x with the block's partial sum of its square (y may be null: the
// norm only).  TS: alpha, b and the arithmetic; TX, TY: storage of x and y.  The row
// padding (flags 0, x 0) gives zeros, so y covers every entry of the vector.
template <typename TS, typename TX, typename TY, bool RESID, int V>
__global__ void __launch_bounds__(256) k_fine(Lvl g, const uint8_t *__restrict__ fl, const TS *__restrict__ al,
                                              const TS *__restrict__ b, const TX *__restrict__ x, TY *__restrict__ y,
                                              double *part, int nb, int sb)
{
    typedef typename Cvt<TS>::C C;
    typedef typename Cvt<TY>::C CY;
    __shared__ double sh[4];
    double acc = 0.0;
    int i, blk;
    const bool on = strip_of(g.Px, nb, sb, i, blk);
    const unsigned plane = (unsigned)g.Py * (unsigned)g.Pz, t = ((unsigned)blk * 256u + threadIdx.x) * V;
    if (on && t < plane) {
        const unsigned q = (unsigned)i * plane + t;
        C v[4][V];
        auto rows = [&](const auto &a, int c) {
            typedef std::decay_t<decltype(a)> A;
            const BoxSten<C, 3, A, true> s{a};
            v[0][c] = s.cell();
            v[1][c] = s.template face<0>(0, 0, 0);
            v[2][c] = s.template face<1>(0, 0, 0);
            v[3][c] = s.template face<2>(0, 0, 0);
        };
#pragma unroll
        for (int c = 0; c < V; c++) rows(FineAcc<TS, TX, V>{fl, x, al, g.S, (long)plane, (long)g.Pz, q, c}, c);
#pragma unroll
        for (int f = 0; f < 4; f++) {
            Vec<TY, V> o;
            Vec<TS, V> bb;
            if (RESID) bb = vat<V>(b + f * g.S, q);
#pragma unroll
            for (int c = 0; c < V; c++) {
                C w = v[f][c];
                if (RESID) {
                    w = Cvt<TS>::ld(bb.get(c)) - w;
                    acc += (double)w * w;
                }
                o.set(c, Cvt<TY>::st((CY)w));
            }
            if (!RESID || y) vput<V>(y + f * g.S, q, o);
        }
    }
    if (RESID && part) {
        for (int o = 32; o > 0; o >>= 1) acc += __shfl_down(acc, o, 64);
        if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = acc;
        __syncthreads();
        if (threadIdx.x == 0) part[blockIdx.x] = sh[0] + sh[1] + sh[2] + sh[3];
    }
}

unsigned fine_blocks(const Lvl &g)  // of an FP64 residual
{
    return strip_grid(g.Px, plane_blocks<double>(g), STRIP);
}
template <typename TS, typename TX, typename TY, bool RESID>
static void launch_fine(const Lvl &g, const uint8_t *fl, const TS *al, const TS *b, const TX *x, TY *y, double *part,
                        hipStream_t s)
{
    const int nb = plane_blocks<TS>(g);
    hipLaunchKernelGGL((k_fine<TS, TX, TY, RESID, lane_nodes<TS>()>), dim3(strip_grid(g.Px, nb, STRIP)), dim3(256), 0, s, g,
                       fl, al, b, x, y, part, nb, STRIP);
}
template <typename TS> void fine_apply(const Lvl &g, const uint8_t *fl, const TS *al, const TS *x, TS *y, hipStream_t s)
{
    launch_fine<TS, TS, TS, false>(g, fl, al, (const TS *)nullptr, x, y, nullptr, s);
}
template <typename TS>
void fine_residual(const Lvl &g, const uint8_t *fl, const TS *al, const TS *b, const TS *x, TS *r, double *part, hipStream_t s)
{
    launch_fine<TS, TS, TS, true>(g, fl, al, b, x, r, part, s);
}
void fine_apply_mixed(const Lvl &g, const uint8_t *fl, const double *al, const float *x, double *y, hipStream_t s)
{
    launch_fine<double, float, double, false>(g, fl, al, (const double *)nullptr, x, y, nullptr, s);
}

// ------------------------------------------- operator on the caller's arrays
//
// y = A x on vectors in the caller's layout (fields concatenated without padding, rows of
// nz, nz, nz and nz + 1 values), FP64, flags and alpha in the node layout: one launch
// where packing x, the operator and unpacking y were three, two of them transposing
// copies of the vector.  Kernel time at 256^3 808 -> 494 us (3.0 TB/s; 444 us in the node
// layout, whose rows are whole lines), 128^3 119 -> 56, 32^3 14 -> 4.7.  A lane takes one
// node: two of them in 16-byte accesses of 8-byte alignment took the same time, other
// block orders 1 to 2% more, fewer registers (6 or 8 waves) two to three times as long.
namespace {
// The node at padded offset q; qa[f]: its index in field f of the caller's vector, whose
// rows and planes are sj[f] and si[f] apart.  A velocity outside its field has a clear
// flag bit, so its read only has to stay inside the vector: before the first entry of
// field f lies field f - 1, behind the last one field f + 1, and with END (the last three
// planes; clamping all of them costs 7%) the last field is clamped.  A pressure outside
// is 0 by position.
template <int DIM, bool END> struct UserAcc {
    typedef double C;
    static constexpr bool MASK = true;
    const uint8_t *fl;
    const double *al, *x[DIM + 1];
    long S, sI, sJ;
    long si[DIM + 1], sj[DIM + 1];
    unsigned q, qa[DIM + 1], end;  // end: last entry of the last field
    bool li, lj, lk, in;           // first node along an axis; a cell of the level

    __device__ __forceinline__ int F(int di, int dj, int dk) const { return at(fl + (di * sI + dj * sJ + dk), q); }
    __device__ __forceinline__ double X(int f, int di, int dj, int dk) const
    {
        if (f == 0) {  // own cell, or the one below along one axis
            const bool off = di < 0 ? li : (dj < 0 ? lj : (dk < 0 ? lk : !in));
            const unsigned d = (unsigned)(-di * (int)si[0] - dj * (int)sj[0] - dk);
            const double v = at(x[0], off ? qa[0] : qa[0] - d);
            return off ? 0.0 : v;
        }
        const long o = di * si[f] + dj * sj[f] + dk;
        if (f < DIM || !END) return at(x[f] + o, qa[f]);
        const int e = (int)qa[f] + (int)o;
        return x[f][e < (int)end ? e : (int)end];
    }
    __device__ __forceinline__ double AL(int d, int di, int dj, int dk) const
    {
        return at(al + d * S + (di * sI + dj * sJ + dk), q);
    }
};

// the rows of node (i, j, k), written to y
template <int DIM, bool END>
__device__ __forceinline__ void user_rows(const Lvl &g, const uint8_t *fl, const double *al, const double *x, double *y,
                                          int i, int j, int k)
{
    UserAcc<DIM, END> a;
    a.fl = fl;
    a.al = al;
    a.S = g.S;
    a.sI = (long)g.Py * g.Pz;
    a.sJ = g.Pz;
    a.q = ((unsigned)i * (unsigned)g.Py + (unsigned)j) * (unsigned)g.Pz + (unsigned)k;
    a.li = i == 0;
    a.lj = j == 0;
    a.lk = k == 0;
    a.in = i < g.nx && j < g.ny && k < g.nz;
    bool own[DIM + 1];
    long off = 0;
#pragma unroll
    for (int f = 0; f <= DIM; f++) {
        const int A = g.nx + (f == 1), B = g.ny + (f == 2), Cc = g.nz + (f == 3);
        a.x[f] = x + off;
        a.si[f] = (long)B * Cc;
        a.sj[f] = Cc;
        a.qa[f] = ((unsigned)i * (unsigned)B + (unsigned)j) * (unsigned)Cc + (unsigned)k;
        own[f] = i < A && j < B && k < Cc;
        if (f == DIM) a.end = (unsigned)((long)A * B * Cc - 1);
        off += (long)A * B * Cc;
    }
    const BoxSten<double, DIM, UserAcc<DIM, END>, DIM == 3> s{a};
    double v[DIM + 1];
    v[0] = s.cell();
    v[1] = s.template face<0>(0, 0, 0);
    v[2] = s.template face<1>(0, 0, 0);
    if constexpr (DIM == 3) v[3] = s.template face<2>(0, 0, 0);
#pragma unroll
    for (int f = 0; f <= DIM; f++)
        if (own[f]) put(y + (a.x[f] - x), a.qa[f], v[f]);
}
}  // namespace

__global__ void __launch_bounds__(256) k_user_apply3(Lvl g, const uint8_t *__restrict__ fl, const double *__restrict__ al,
                                                     const double *__restrict__ x, double *__restrict__ y, int nb, int sb)
{
    int i, blk;
    if (!strip_of(g.Px, nb, sb, i, blk)) return;
    const unsigned t = (unsigned)blk * 256u + threadIdx.x;
    if (t >= (unsigned)g.Py * (unsigned)g.Pz) return;
    const int j = (int)(t / (unsigned)g.Pz), k = (int)(t - (unsigned)j * (unsigned)g.Pz);
    if (k > g.nz) return;
    if (i < g.nx - 2) user_rows<3, false>(g, fl, al, x, y, i, j, k);
    else user_rows<3, true>(g, fl, al, x, y, i, j, k);
}
__global__ void __launch_bounds__(256) k_user_apply2(Lvl g, const uint8_t *__restrict__ fl, const double *__restrict__ al,
                                                     const double *__restrict__ x, double *__restrict__ y)
{
    const unsigned n = blockIdx.x * 256u + threadIdx.x;
    if (n >= (unsigned)g.S) return;
    const int i = (int)(n / (unsigned)g.Py);
    user_rows<2, true>(g, fl, al, x, y, i, (int)(n - (unsigned)i * (unsigned)g.Py), 0);
}
void user_apply(const Lvl &g, const uint8_t *fl, const double *al, const double *x, double *y, hipStream_t s)
{
    if (g.dim == 2) {
        hipLaunchKernelGGL(k_user_apply2, dim3((unsigned)((g.S + 255) / 256)), dim3(256), 0, s, g, fl, al, x, y);
        return;
    }
    const int nb = (int)(((long)g.Py * g.Pz + 255) / 256), sb = nb < STRIP ? nb : STRIP;
    hipLaunchKernelGGL(k_user_apply3, dim3(strip_grid(g.Px, nb, sb)), dim3(256), 0, s, g, fl, al, x, y, nb, sb);
}

#define INST_F(T)                                                                                          \
    template void fine_apply<T>(const Lvl &, const uint8_t *, const T *, const T *, T *, hipStream_t);     \
    template void fine_residual<T>(const Lvl &, const uint8_t *, const T *, const T *, const T *, T *, double *, hipStream_t);
INST_F(double)
INST_F(float)
INST_F(bf16)

}  // namespace st
