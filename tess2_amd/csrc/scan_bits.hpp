// scan_bits.hpp -- one scan line of the reference's cell scan from the
// line's PtInCell verdicts held as bits.  Header-only and free of device
// intrinsics, so that a host build can check it against the point-by-point
// walk.
#pragma once

namespace t2 {

__host__ __device__ __forceinline__ int row_high(unsigned long long r)
{
    return 63 - __builtin_clzll(r);
}
__host__ __device__ __forceinline__ int row_high(unsigned r) { return 31 - __builtin_clz(r); }
__host__ __device__ __forceinline__ int row_low(unsigned long long r)
{
    return __builtin_ffsll((long long)r) - 1;
}
__host__ __device__ __forceinline__ int row_low(unsigned r) { return __builtin_ffs((int)r) - 1; }

// The reference's two x walks along one scan line (src/dense.cpp:1546-1620)
// from the line's verdict bits (bit x = PtInCell at x, n0 points, at most the
// word's bits): each
// walk moves one point at a time until the verdict changes, so it ends at the
// nearest bit of the other value, found here with one bit scan.
//   left walk from x0 = x_left: inside -> down through the run (x_left = the
//     first point outside, unchanged when the run reaches 0); outside -> up
//     to the first inside point (x_left = it)
//   right walk from x_right: x0 inside -> up through the run if x_right is
//     inside (x_right = the first point outside); x0 outside -> down to the
//     first inside point at or below x_right (x_right = it)
template <class W>
__host__ __device__ __forceinline__ void walk_row_word(W row, int n0, int &x_left, int &x_right,
                                                       int &min_xi, int &max_xi)
{
    constexpr W ONE = 1;
    const W all = n0 >= (int)(8 * sizeof(W)) ? ~(W)0 : (W)((ONE << n0) - ONE);
    const int x0 = x_left, xr = x_right;
    const bool x_in = (row >> x0) & ONE;
    if (x_in) {
        const W out = ~row & ((ONE << x0) - ONE);   // outside, below x0
        int lo = 0;
        if (out) {
            lo = row_high(out) + 1;   // one above the highest outside point
            x_left = lo - 1;
        }
        min_xi = lo;
        max_xi = x0;
        if ((row >> xr) & ONE) {
            const W outr = ~row & all & ~(((ONE + ONE) << xr) - ONE);   // outside, above xr
            int hi = n0 - 1;
            if (outr) {
                x_right = row_low(outr);
                hi = x_right - 1;
            }
            min_xi = min_xi < xr ? min_xi : xr;
            max_xi = max_xi > hi ? max_xi : hi;
        }
    } else {
        const W inl = row & ~(((ONE + ONE) << x0) - ONE);   // inside, above x0
        if (inl) {
            const int xa = row_low(inl);
            x_left = xa;
            min_xi = xa;
            max_xi = xa;
        }
        const W inr = row & (((ONE + ONE) << xr) - ONE);    // inside, at or below xr
        if (inr) {
            const int xb = row_high(inr);
            x_right = xb;
            min_xi = min_xi < xb ? min_xi : xb;
            max_xi = max_xi > xb ? max_xi : xb;
        }
    }
}

__host__ __device__ __forceinline__ void walk_row_bits(unsigned long long row, int n0,
                                                       int &x_left, int &x_right, int &min_xi,
                                                       int &max_xi)
{
    walk_row_word<unsigned long long>(row, n0, x_left, x_right, min_xi, max_xi);
}

// lines of at most 32 points in one 32-bit word
__host__ __device__ __forceinline__ void walk_row_bits32(unsigned row, int n0, int &x_left,
                                                         int &x_right, int &min_xi, int &max_xi)
{
    walk_row_word<unsigned>(row, n0, x_left, x_right, min_xi, max_xi);
}

}  // namespace t2
