// The steps of a key switch, a rescale and the operations around them as first loads and last stores of line transforms (ntt_fine.hpp).
#pragma once
#include "conv_core.hpp"
#include "ntt_fine.hpp"

namespace ckks {

// A pointer to tables that no launch writes: loads of uniform entries through it are scalar loads wherever they stand (behind a
// store the compiler would otherwise fetch them through the vector memory pipe, whose waits also wait for the data requested before).
template <class T>
__device__ __forceinline__ const T* table_ptr(const T* p) {
    return (const T*)(const __attribute__((address_space(4))) T*)(uintptr_t)p;
}

// ---- inverse transforms of a ciphertext's polynomials: where the input comes from ----
struct LoadFrom {                // limb j of src, left as it is
    const u64* src;
    long N;
    template <class AR, int R>
    __device__ __forceinline__ void adjacent(const AR& ar, const LimbRef& l, unsigned p, typename AR::V (&v)[R]) const {
        u64 x[R];
        load_adjacent(src + (long)l.j * N + p, x);
#pragma unroll
        for (int j = 0; j < R; j++) v[j] = ar.from_canonical(x[j]);
    }
};
struct LoadReversed {            // limb j of src read backwards (X -> X^-1 in the NTT domain, poly_arithmetic.cuh:666-680)
    const u64* src;
    long N;
    template <class AR, int R>
    __device__ __forceinline__ void adjacent(const AR& ar, const LimbRef& l, unsigned p, typename AR::V (&v)[R]) const {
        u64 x[R];
        load_adjacent(src + (long)l.j * N + (N - R - p), x);
#pragma unroll
        for (int j = 0; j < R; j++) v[j] = ar.from_canonical(x[R - 1 - j]);
    }
};
struct LoadProduct {             // limb j of a times limb j of b (the a1 a2 term of a product, poly_arithmetic.cuh:787-824)
    const u64 *a, *b;
    long N;
    template <class AR, int R>
    __device__ __forceinline__ void adjacent(const AR& ar, const LimbRef& l, unsigned p, typename AR::V (&v)[R]) const {
        u64 x[R], y[R];
        load_adjacent(a + (long)l.j * N + p, x);
        load_adjacent(b + (long)l.j * N + p, y);
#pragma unroll
        for (int j = 0; j < R; j++) v[j] = ar.settle(ar.mulmod(ar.from_canonical(x[j]), ar.from_canonical(y[j])));
    }
};

// ---- forward transform of the digits over T: the conversion Q_j -> T (BasisConv.cuh:84-179) at the values the first round takes ----
// limb (digit y, T prime j); sources below 2^50
template <int MAXS>
struct LoadDigits {
    const u64* in;               // l + 1 limbs, coefficient domain
    const ConvBlock* blocks;     // one per digit
    const PrimeConst* primes;
    long N;
    template <class AR, int R>
    __device__ __forceinline__ void gather(const AR& ar, const LimbRef& l, const unsigned (&pos)[R], typename AR::V (&v)[R]) const {
        const ConvBlock& b = *table_ptr(blocks + l.y);
        const PrimeConst* pr = table_ptr(primes);
        const u64 neg_dmod = ar.q - b.dmod[l.j];
        constexpr int H = MAXS <= 2 ? R : 4;                     // values in work together
#pragma unroll
        for (int j0 = 0; j0 < R; j0 += H) {
            u64 x[H][MAXS];
#pragma unroll
            for (int j = 0; j < H; j++)
#pragma unroll
                for (int s = 0; s < MAXS; s++) x[j][s] = in[(long)b.src_limb[s] * N + pos[j0 + j]];
#pragma unroll
            for (int j = 0; j < H; j++) {
                u64 y[MAXS];
                double yd[MAXS];
                conv_scale<MAXS, CONV_SRC_F64>(x[j], b, pr, y, yd);
                v[j0 + j] = conv_columns(y, b.hat[l.j], conv_quotient(yd, b, pr), neg_dmod).reduce(ar);
            }
        }
    }
};

// ---- inverse transform of the sums over T: the external product with the key (ExternalProduct.cuh:56-83) at the values it starts from ----
// limb (polynomial z, output block y, T prime j)
struct LoadExternal {
    const u64* up;               // digits: limb d * t_num + j
    const u64* key;              // limb z * key_z + d * key_digit + y * t_num + j
    long N, key_digit, key_z;    // strides in limbs
    int t_num, ndigits;
    template <class AR, int R>
    __device__ __forceinline__ void adjacent(const AR& ar, const LimbRef& l, unsigned p, typename AR::V (&v)[R]) const {
        const u64* cp = up + (long)l.j * N + p;
        const u64* kp = key + ((long)l.z * key_z + (long)l.y * t_num + l.j) * N + p;
        const long cs = (long)t_num * N, ks = key_digit * N;
        constexpr int H = R < 4 ? R : 4;                         // words at a time: their sums and two digits' words fit the registers
#pragma unroll
        for (int j0 = 0; j0 < R; j0 += H) {
            PmSum acc[H];
            u64 x[H], k[H];
            load_adjacent<H>(cp + j0, x);
            load_adjacent<H>(kp + j0, k);
            for (int d = 0; d < ndigits; d++) {
                u64 xn[H], kn[H];
                const long at = d + 1 < ndigits ? d + 1 : d;      // one digit ahead (the last one once more)
                load_adjacent<H>(cp + at * cs + j0, xn);
                load_adjacent<H>(kp + at * ks + j0, kn);
#pragma unroll
                for (int j = 0; j < H; j++) acc[j].add(x[j], k[j]);
                if ((d & 7) == 7) {
#pragma unroll
                    for (int j = 0; j < H; j++) acc[j].renormalise(ar);
                }
#pragma unroll
                for (int j = 0; j < H; j++) { x[j] = xn[j]; k[j] = kn[j]; }
            }
#pragma unroll
            for (int j = 0; j < H; j++) v[j0 + j] = acc[j].reduce(ar);
        }
    }
};

// ---- forward transform of the results: what happens to them on the way out (limb (polynomial y, modulus j)) ----
struct StoreAddProducts {        // + a1 b2 + a2 b1 (polynomial 0), + b1 b2 (polynomial 1): the rest of a product of two ciphertexts
    const u64 *a1, *b1, *a2, *b2;
    long N;
    template <class AR, int R>
    __device__ __forceinline__ void adjacent(const AR& ar, const LimbRef& l, unsigned p, const typename AR::V (&v)[R]) const {
        const long at = (long)l.j * N + p;
        u64 x[R], y[R];
        typename AR::V t[R];
        if (l.y == 0) {
            load_adjacent(a1 + at, x);
            load_adjacent(b2 + at, y);
#pragma unroll
            for (int j = 0; j < R; j++) t[j] = v[j] + ar.mulmod(ar.from_canonical(x[j]), ar.from_canonical(y[j]));
            load_adjacent(a2 + at, x);
            load_adjacent(b1 + at, y);
        } else {
#pragma unroll
            for (int j = 0; j < R; j++) t[j] = v[j];
            load_adjacent(b1 + at, x);
            load_adjacent(b2 + at, y);
        }
#pragma unroll
        for (int j = 0; j < R; j++) x[j] = ar.to_canonical_fwd(t[j] + ar.mulmod(ar.from_canonical(x[j]), ar.from_canonical(y[j])));
        store_adjacent(l.ptr + p, x);
    }
};
// (polynomial 1: + b) through the slot permutation i -> bitrev(((pow (2 bitrev(i) + 1) mod 2N) - 1) / 2) (KeySwitch_23.cuh:582-585): eight
// adjacent slots go to eight adjacent slots in another order, so a lane stores within one aligned 64-byte piece
struct StoreRotated {
    u64* out;
    const u64* b;
    u64 pow;
    long N, out_poly_stride;     // words between the polynomials of out
    int logN;
    template <class AR, int R>
    __device__ __forceinline__ void adjacent(const AR& ar, const LimbRef& l, unsigned p, const typename AR::V (&v)[R]) const {
        u64 x[R];
        if (l.y == 1) load_adjacent(b + (long)l.j * N + p, x);
        u64* dst = out + (long)l.y * out_poly_stride + (long)l.j * N;
        const unsigned mask = (2u << logN) - 1u, pw = (unsigned)pow;
#pragma unroll
        for (int j = 0; j < R; j++) {
            u64 w = ar.to_canonical_fwd(v[j]);
            if (l.y == 1) w = csub(w + x[j], ar_q(ar));
            const unsigned e = 2u * (__brev(p + j) >> (32 - logN)) + 1u;
            dst[__brev((((pw * e) & mask) - 1u) >> 1) >> (32 - logN)] = w;
        }
    }
    template <class AR> static __device__ __forceinline__ u64 ar_q(const AR& ar) { return (u64)ar.q; }
};
struct StoreAddReversed {        // polynomial 1: + b read backwards (KeySwitch_23.cuh:454, 467)
    const u64* b;
    long N;
    template <class AR, int R>
    __device__ __forceinline__ void adjacent(const AR& ar, const LimbRef& l, unsigned p, const typename AR::V (&v)[R]) const {
        u64 w[R], x[R];
        if (l.y == 1) load_adjacent(b + (long)l.j * N + (N - R - p), x);
#pragma unroll
        for (int j = 0; j < R; j++) {
            w[j] = ar.to_canonical_fwd(v[j]);
            if (l.y == 1) w[j] = csub(w[j] + x[R - 1 - j], (u64)ar.q);
        }
        store_adjacent(l.ptr + p, w);
    }
};

// ---- rescale (Scheme_23.cuh:321-367): limb l modulo the prime of the limb in work; (c - x) q_l^-1 on the way out ----
struct LoadReduced {
    const u64* src;              // limb l of polynomial y at src + y * poly_stride
    long poly_stride;
    template <class AR, int R>
    __device__ __forceinline__ void gather(const AR& ar, const LimbRef& l, const unsigned (&pos)[R], typename AR::V (&v)[R]) const {
        const u64* s = src + (long)l.y * poly_stride;
        u64 x[R];
#pragma unroll
        for (int j = 0; j < R; j++) x[j] = s[pos[j]];
#pragma unroll
        for (int j = 0; j < R; j++) v[j] = ar.balance(exact_u2d(x[j]));
    }
};
struct StoreRescaled {
    u64* cipher;                 // limb j of polynomial y at cipher + y * poly_stride + j * N
    const u64* inv;              // q_l^-1 mod q_j
    long poly_stride, N;
    template <class AR, int R>
    __device__ __forceinline__ void adjacent(const AR& ar, const LimbRef& l, unsigned p, const typename AR::V (&v)[R]) const {
        u64* c = cipher + (long)l.y * poly_stride + (long)l.j * N + p;
        u64 x[R];
        load_adjacent(c, x);
        const double w = ar.from_canonical(table_ptr(inv)[l.j]);         // balanced for wide primes: the product's quotient estimate needs it
#pragma unroll
        for (int j = 0; j < R; j++) x[j] = ar.canon(ar.mulmod(exact_u2d(x[j]) - ar.balance(v[j]), w));      // |c - x| < 1.5 q
        store_adjacent(c, x);
    }
};

}  // namespace ckks
