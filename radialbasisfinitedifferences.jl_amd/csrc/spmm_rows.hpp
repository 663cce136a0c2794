// spmm_rows.hpp -- a CSR row times 8 fields, 16 lanes a row: the sum shared by
// the plain products, the plan's products and the RK stages.
#pragma once
#include <type_traits>

#include "device_common.hpp"

namespace rbffd {

// Lane L of each 16-lane DPP row, in the lanes of bank BANK (4 lanes a bit) of
// that row; the other lanes keep old.
template <int L, int BANK>
__device__ __forceinline__ int row_bcast_bank(int old, int v)
{
    return __builtin_amdgcn_update_dpp(old, v, 0x150 + L, 0xF, BANK, false);
}
template <int L, int BANK>
__device__ __forceinline__ double row_bcast_bank(double old, double v)
{
    return __longlong_as_double(__builtin_amdgcn_update_dpp(__double_as_longlong(old), __double_as_longlong(v),
                                                            0x150 + L, 0xF, BANK, false));
}

// Entries 4 T .. 4 T + 3 of a block of 32, 16 to a register, one to each quad of
// lanes.
template <int T, typename V>
__device__ __forceinline__ V spread_entry(const V (&a)[2])
{
    constexpr int r = T / 4, l = 4 * (T % 4);
    V v = row_bcast_bank<l, 0x1>(a[r], a[r]);
    v = row_bcast_bank<l + 1, 0x2>(v, a[r]);
    v = row_bcast_bank<l + 2, 0x4>(v, a[r]);
    return row_bcast_bank<l + 3, 0x8>(v, a[r]);
}

template <int T, int N, class Fn>
__device__ __forceinline__ void for_steps(Fn &&f)
{
    if constexpr (T < N) {
        f(std::integral_constant<int, T>{});
        for_steps<T + 1, N>(f);
    }
}

// A row's entries b .. b + 31, 16 a load, entry b + j in lane j % 16, register j /
// 16; zeros past the row's end.  c: the column, or its place in a plan's list.
// (Two entries a lane, in one load each of columns and values, took 5 us more a
// million rows of 31: most of those loads start off their width.)
struct RowEntries {
    int c[2];
    double v[2];
};

template <typename TV, typename TC>
__device__ __forceinline__ RowEntries row_entries(const TV *val, const TC *col, int len, int b)
{
    RowEntries e;
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        const int j = b + 16 * r + (int)(threadIdx.x & 15);
        e.c[r] = 0;
        e.v[r] = 0.0;
        if (j < len) {
            e.c[r] = (int)col[j];
            e.v[r] = (double)val[j];
        }
    }
    return e;
}

// most: the largest len of the wavefront's four rows; full: all have it.
__device__ __forceinline__ void rows_extent(int len, int &most, bool &full)
{
    most = max(max(__builtin_amdgcn_readlane(len, 0), __builtin_amdgcn_readlane(len, 16)),
               max(__builtin_amdgcn_readlane(len, 32), __builtin_amdgcn_readlane(len, 48)));
    full = __builtin_amdgcn_ballot_w64(len == most) == ~0ull;
}

// acc = the sum over j < len of val[j] x(at(col[j])) for this lane's two fields, 2
// (lane % 4) and the next, in every quad of the row's 16 lanes.  val, col: the
// row's entries; len: its length (0 for a group without a row); most, full: as
// rows_extent (most may exceed every len); x: node 0's row.  Padded entries read
// node at(0) where the wavefront has any entry, and are dropped whatever it holds.
//
// Loads are bound by the address unit, which takes a quad of lanes a cycle
// whatever they carry (with two lanes of 32 bytes it was busy 87% of 185 us over a
// million rows, n = 31, and is 88% of 134 now).  So an entry's 64 bytes of x go to one quad, 16 bytes a lane,
// and columns and values come in once, 16 entries a load, and DPP broadcasts
// hand entry j to its quad: 1.5 cycles an entry against 2 with two lanes of 32
// bytes and a column and a value loaded by each.  All gathers of up to 32
// entries are in flight together: two or four rows a lane group were slower.
// Quad k sums entries k, k + 4, ... in order; the quads are added by rotations.
template <typename TV, typename TC, class At>
__device__ __forceinline__ void row_times_8(double (&acc)[2], const TV *val, const TC *col, int len, int most,
                                            bool full, const double *x, At &&at)
{
    constexpr int STEPS = 8;
    const int quad = (threadIdx.x & 15) / 4;
    const double *const xf = x + 2 * (threadIdx.x & 3);
    acc[0] = acc[1] = 0.0;
    for (int b = 0; b < most; b += 32) {
        RowEntries e = row_entries(val, col, len, b);
#pragma unroll
        for (int r = 0; r < 2; ++r) e.c[r] = at(e.c[r]);
        // one path for the loads of padded entries and real ones: with two,
        // every gather would wait for the one before
        double xv[STEPS][2];
        for_steps<0, STEPS>([&](auto tc) {
            constexpr int t = decltype(tc)::value;
            if (b + 4 * t < most) {  // uniform
                const double *const p = xf + 8L * spread_entry<t>(e.c);
                xv[t][0] = p[0];
                xv[t][1] = p[1];
            }
        });
        for_steps<0, STEPS>([&](auto tc) {
            constexpr int t = decltype(tc)::value;
            const int j = b + 4 * t;
            if (j < most) {
                const double vj = spread_entry<t>(e.v);
                const bool part = !full || j + 4 > most;  // uniform
#pragma unroll
                for (int f = 0; f < 2; ++f) {
                    double xf = xv[t][f];
                    if (part) xf = j + quad < len ? xf : 0.0;
                    acc[f] = __builtin_fma(vj, xf, acc[f]);
                }
            }
        });
    }
#pragma unroll
    for (int f = 0; f < 2; ++f) {
        acc[f] += dpp_f64<0x120 | 4>(acc[f]);  // row_ror
        acc[f] += dpp_f64<0x120 | 8>(acc[f]);
    }
}

// What becomes of a row's sum.  MODE 0: y = alpha A x + beta y; MODE 1: one
// Shu-Osher stage y = a u + b x + c (A x), rows with fixed[r] != 0 keeping u (y may
// be u: the same lane reads and writes a value).
struct RowsOut {
    double *y;
    double alpha, beta;
    const double *u;
    const uint8_t *fixed;
    double a, b, c;
};

// the two fields of a row of 8 that this lane holds (the first quad's lanes)
template <int MODE>
__device__ __forceinline__ void put_row_8(const RowsOut &o, long row, const double (&acc)[2], const double *x)
{
    const long e = row * 8 + 2 * (threadIdx.x & 3);
    const bool hold = MODE == 1 && o.fixed && o.fixed[row];
#pragma unroll
    for (int f = 0; f < 2; ++f) {
        if constexpr (MODE == 0) {
            double r = o.alpha * acc[f];
            if (o.beta != 0.0) r = __builtin_fma(o.beta, o.y[e + f], r);
            o.y[e + f] = r;
        } else {
            const double ui = o.u[e + f];
            o.y[e + f] = hold ? ui : o.a * ui + o.b * x[e + f] + o.c * acc[f];
        }
    }
}

}  // namespace rbffd
