// mnc_orbit.h -- the quadrature's reflection symmetry, used by the FP64 Newton
// kernel (mnc_rows.hip) and by the host code that builds its tables.
//
// The nodes come in orbits of four, (+-xi, +-eta) with equal weights (2Q
// equispaced azimuths (j + 1/2) pi / Q, Q even: no node is its own mirror
// image).  Every moment is even or odd under each reflection:
//   cos(m phi): even in eta, odd in xi when m is odd;
//   sin(m phi): odd in eta, odd in xi when m is even.
// With the class of moment k as two bits (1: odd in xi, 2: odd in eta), the
// four exponents alpha.m of an orbit are signed sums of four partial sums, one
// per class, and with w e at the four points combined into
//   C[c] = sum over the orbit of sign_c w e
// (sign_c the sign of class c at the point) the sums over the quadrature are
// sums over orbits:  sum w e m_i m_j = sum_orbits C[cls_i ^ cls_j] m_i m_j,
// m at the orbit's point with xi, eta > 0: a quarter of the products.
#pragma once

#ifndef __HIPCC__
#define MNC_HD
#else
#define MNC_HD __host__ __device__
#endif

namespace mnc {

MNC_HD constexpr int orbit_nm(int N) { return (N + 1) * (N + 2) / 2; }

// class of moment k in the order l = 0.., m = -l..l with l + m even
MNC_HD constexpr int orbit_class(int k) {
    int i = 0;
    for (int l = 0;; ++l)
        for (int m = -l; m <= l; ++m) {
            if ((l + m) & 1) continue;
            if (i++ != k) continue;
            const int odd = (m < 0 ? -m : m) & 1;
            return m >= 0 ? odd : 2 | (odd ^ 1);
        }
}

// moments of order N in class c
MNC_HD constexpr int orbit_class_size(int N, int c) {
    int n = 0;
    for (int k = 0; k < orbit_nm(N); ++k) n += orbit_class(k) == c;
    return n;
}

// The sign of class c at image `img` of an orbit (bit 1: -xi, bit 2: -eta) is
// negative when they share an odd number of bits.
MNC_HD constexpr bool orbit_negative(int c, int img) { return ((c & img & 1) ^ ((c & img) >> 1)) != 0; }

// The sums of one solve in the order the kernel forms them, class by class.
// Direct Hessian: entry e is the product m_a m_b (a >= b within a class; for
// two classes a runs over the smaller one, so that C m_a is formed least
// often).  Gaunt form: entry e is the order-2N moment a.
template <int N, bool GAUNT>
struct OrbitSums {
    static constexpr int n = orbit_nm(N), n2 = orbit_nm(2 * N);
    static constexpr int count = GAUNT ? n2 : n * (n + 1) / 2;
    struct Lists {
        int first[5];
        unsigned char a[count], b[count], cls[n2];
    };
    MNC_HD static constexpr Lists lists() {
        Lists L{};
        for (int k = 0; k < n2; ++k) L.cls[k] = (unsigned char)orbit_class(k);
        int e = 0;
        for (int c = 0; c < 4; ++c) {
            L.first[c] = e;
            if (GAUNT) {
                for (int k = 0; k < n2; ++k)
                    if (L.cls[k] == c) { L.a[e] = (unsigned char)k; L.b[e++] = 0; }
            } else if (c == 0) {
                for (int p = 0; p < 4; ++p)
                    for (int i = 0; i < n; ++i)
                        for (int j = 0; j <= i; ++j)
                            if (L.cls[i] == p && L.cls[j] == p) { L.a[e] = (unsigned char)i; L.b[e++] = (unsigned char)j; }
            } else {
                for (int p = 0; p < 4; ++p) {
                    const int q = p ^ c;
                    if (q < p) continue;
                    int np = 0, nq = 0;
                    for (int i = 0; i < n; ++i) { np += L.cls[i] == p; nq += L.cls[i] == q; }
                    const int s = np <= nq ? p : q, o = np <= nq ? q : p;
                    for (int i = 0; i < n; ++i)
                        for (int j = 0; j < n; ++j)
                            if (L.cls[i] == s && L.cls[j] == o) { L.a[e] = (unsigned char)i; L.b[e++] = (unsigned char)j; }
                }
            }
        }
        L.first[4] = e;
        return L;
    }
};

// Where the kernel keeps sum e of class c in its buffer: the closure without a
// separate gradient (Mn) carries sum w e right after the class 0 sums.
MNC_HD constexpr int orbit_slot(int e, int c, bool ppn) { return e + (!ppn && c > 0 ? 1 : 0); }

}  // namespace mnc
