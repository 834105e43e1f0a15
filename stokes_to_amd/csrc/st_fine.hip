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
//   y = A x           540 -> 444  262 -> 228   88 -> 68  35 -> 27   31 -> 10  24 -> 10
//   r = b - A x       627 -> 515  316 -> 249  101 -> 74  44 -> 33   36 -> 13  28 -> 11
// At 256^3 that is 3.7 to 4.6 TB/s of HBM traffic (FP32 0.83 / 1.14 GB, near the least).
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
    *reinterpret_cast<typename Vec<T, N>::R *>(reinterpret_cast<char *>(p) + i * (unsigned)sizeof(T)) = x.v;
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

#define INST_F(T)                                                                                          \
    template void fine_apply<T>(const Lvl &, const uint8_t *, const T *, const T *, T *, hipStream_t);     \
    template void fine_residual<T>(const Lvl &, const uint8_t *, const T *, const T *, const T *, T *, double *, hipStream_t);
INST_F(double)
INST_F(float)
INST_F(bf16)

}  // namespace st
