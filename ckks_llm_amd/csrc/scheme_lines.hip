// The client's transforms with the step before or behind them inside (ntt_fine.hpp): encoding, both halves of an encryption, and the
// way back to coefficients that a decoding starts with.
//
// As launches of their own the steps around the transforms wrote every sampled or encoded limb to memory for the transform to read it
// back, and at these sizes a launch costs as much as the step: encode 2 -> 1 launches, encrypt 4 -> 2, decode 3 -> 2.
// Encode, encrypt, decrypt, decode of ten limbs of 2^14: kernels 82 -> 50 us (encode 11.5 -> 8.0, encryption 32 -> 22, decoding 36 -> 16).
#include "ks_ops.hpp"
#include "samplers.hpp"

namespace ckks {

// values times the scale, truncated, modulo the limb's prime (Encoder.cuh:75): the 64-bit integer is hi 2^32 + lo
struct LoadEncoded {
    const double* vals;
    double scale;
    template <class AR, int R>
    __device__ __forceinline__ void gather(const AR& ar, const LimbRef&, const unsigned (&pos)[R], typename AR::V (&v)[R]) const {
        double x[R];
#pragma unroll
        for (int j = 0; j < R; j++) x[j] = vals[pos[j]];
        const double c32 = ar.balance(4294967296.0);
#pragma unroll
        for (int j = 0; j < R; j++) {
            const long long d = (long long)(x[j] * scale);
            v[j] = ar.balance((double)(unsigned)d + ar.mulmod((double)(int)(d >> 32), c32));
        }
    }
};
struct LoadTernary {             // one byte per coefficient: 0 below 128, 1 below 192, -1 above (Sampler_impl.cuh:96-113 at probability 1/2)
    const uint8_t* random;
    template <class AR, int R>
    __device__ __forceinline__ void gather(const AR&, const LimbRef&, const unsigned (&pos)[R], typename AR::V (&v)[R]) const {
        unsigned b[R];
#pragma unroll
        for (int j = 0; j < R; j++) b[j] = random[pos[j]];
#pragma unroll
        for (int j = 0; j < R; j++) v[j] = b[j] < 128 ? 0.0 : b[j] < 192 ? 1.0 : -1.0;
    }
};
struct LoadGaussian {            // one word per coefficient, polynomial y at words + y N
    const uint32_t* words;
    long N;
    GaussSteps g;
    template <class AR, int R>
    __device__ __forceinline__ void gather(const AR&, const LimbRef& l, const unsigned (&pos)[R], typename AR::V (&v)[R]) const {
        uint32_t u[R];
#pragma unroll
        for (int j = 0; j < R; j++) u[j] = words[(long)l.y * N + pos[j]];
#pragma unroll
        for (int j = 0; j < R; j++) v[j] = (double)gauss_value(u[j], g);
    }
};
struct StoreEncrypted {          // + v pk.a (polynomial 0), + v pk.b + m (polynomial 1) (Scheme_23.cuh:92-111)
    const u64 *v, *pk, *mx;      // limb j of v at v + j N; pk as the ciphertext; mx may be null
    long N, pk_poly_stride;
    template <class AR, int R>
    __device__ __forceinline__ void adjacent(const AR& ar, const LimbRef& l, unsigned p, const typename AR::V (&e)[R]) const {
        const long at = (long)l.j * N + p;
        u64 x[R], y[R], m[R];
        load_adjacent(v + at, x);
        load_adjacent(pk + (long)l.y * pk_poly_stride + at, y);
        const bool add = l.y == 1 && mx;
        if (add) load_adjacent(mx + at, m);
#pragma unroll
        for (int j = 0; j < R; j++) x[j] = ar.to_canonical_fwd(e[j] + ar.mulmod(ar.from_canonical(x[j]), ar.from_canonical(y[j])));
        if (add) {
#pragma unroll
            for (int j = 0; j < R; j++) x[j] = csub(x[j] + m[j], (u64)ar.q);
        }
        store_adjacent(l.ptr + p, x);
    }
};

// N = 2^12 .. 2^15 and all Q primes of the level on one FP64 back end: at 2^16 the transforms of ntt.hip with their compact values between
// the passes are the faster ones, and integer primes have no small signed inputs.
static bool client_lines_apply(const ckks_ctx* c, int l, int* back_end) {
    if (c->ks_split || c->arith_mode != 0 || c->ntt_mode != 0 || c->ntt_fine == 4 || c->ev_mid_armed || c->logN < 12 || c->logN > 15) return false;
    const int be = ntt_back_end(c, c->K);
    if (be > 1) return false;
    for (int i = 0; i <= l; i++)
        if (ntt_back_end(c, c->K + i) != be) return false;
    *back_end = be;
    return true;
}

int launch_encode_lines(ckks_ctx* c, uint64_t* mx, const double* vals, long scale, int l, bool* done) {
    int be = 0;
    *done = client_lines_apply(c, l, &be) && words16({mx});
    if (!*done) return CKKS_OK;
    const NttArgs a = line_args(c, (u64*)mx, false, c->K, 1, l + 1, c->L + 1, 0);
    const LoadEncoded ld{vals, (double)scale};
    return be == 0 ? launch_lines<F64Arith, false>(c, a, l + 1, 0, ld, StoreLimb()) : launch_lines<F64WideArith, false>(c, a, l + 1, 1, ld, StoreLimb());
}
int launch_encrypt_lines(ckks_ctx* c, uint64_t* cipher, const uint64_t* mx, const uint64_t* pk, const uint8_t* random, uint64_t* scratch, int l, bool* done) {
    int be = 0;
    *done = client_lines_apply(c, l, &be) && words16({cipher, mx, pk, scratch});
    if (!*done) return CKKS_OK;
    const long N = c->N, L1 = c->L + 1;
    const NttArgs va = line_args(c, (u64*)scratch, false, c->K, 1, l + 1, l + 1, 0), ea = line_args(c, (u64*)cipher, false, c->K, 2, l + 1, L1, 0);
    const LoadTernary lv{random};
    const LoadGaussian le{(const uint32_t*)(random + N), N, gauss_steps()};
    const StoreEncrypted st{(const u64*)scratch, (const u64*)pk, (const u64*)mx, N, N * L1};
    if (be == 0) {
        if (int rc = launch_lines<F64Arith, false>(c, va, l + 1, 0, lv, StoreLimb())) return rc;
        return launch_lines<F64Arith, false>(c, ea, 2 * (l + 1), 0, le, st);
    }
    if (int rc = launch_lines<F64WideArith, false>(c, va, l + 1, 1, lv, StoreLimb())) return rc;
    return launch_lines<F64WideArith, false>(c, ea, 2 * (l + 1), 1, le, st);
}
// limbs 0 .. l of mx as coefficients in out, mx left as it is
int launch_coefficients_lines(ckks_ctx* c, uint64_t* out, const uint64_t* mx, int l, bool* done) {
    int be = 0;
    *done = client_lines_apply(c, l, &be) && words16({out, mx});
    if (!*done) return CKKS_OK;
    const NttArgs a = line_args(c, (u64*)out, true, c->K, 1, l + 1, l + 1, 0);
    const LoadFrom ld{(const u64*)mx, c->N};
    return be == 0 ? launch_lines<F64Arith, true>(c, a, l + 1, 0, ld, StoreLimb()) : launch_lines<F64WideArith, true>(c, a, l + 1, 1, ld, StoreLimb());
}

}  // namespace ckks
