// Transforms of small batches and small rings with eight values per lane (ntt_lines.hpp): whole limbs in one workgroup where a
// limb fits LDS, otherwise the two passes of ntt.hip on twice the lanes, in one paired launch (pair_run.hpp) or in two launches.
// Same words as every other form.
#include <type_traits>

#include "ntt_lines.hpp"

namespace ckks {

PairArgs pair_args(const ckks_ctx* c, int limbs);
unsigned pair_blocks(int limbs, unsigned tiles);

constexpr int FINE_RL = 3;

// SHARED: the tile is one half of a paired launch - what it hands to or takes from the other pass moves as shared accesses
template <class AR, int SA, int SB, bool INVERSE, bool SHARED>
__device__ __forceinline__ void fine_strided_tile(u64* limb, unsigned tile, const typename AR::TW* __restrict__ tw, const AR& ar, typename AR::V* lds,
                                                  const TileClaim& claim = TileClaim()) {
    typedef FineStrided<SA, SB, FINE_RL> F;
    constexpr int RL = FINE_RL, R = 1 << RL, C0 = line_first<SA, RL>();
    constexpr long N2 = 1l << SB;
    const unsigned cl = threadIdx.x % F::CW, u = threadIdx.x / F::CW;
    u64* col = limb + tile * F::CW + cl;
    auto at = [&](unsigned p) { return lds + p * F::CW + cl; };
    typedef LineRound<SA, RL, 0, C0> LR;
    typename AR::V v[R];
    u64 x[R];
    if constexpr (!INVERSE) {
        RoundTw<AR, SA, RL, 0, C0> w;
        w.load(tw, 1u, u);
#pragma unroll
        for (int h = 0; h < LR::GROUPS; h++)
#pragma unroll
            for (int j = 0; j < (1 << C0); j++) x[(h << C0) + j] = col[LR::pos(LR::group(u, h), j) * N2];
        const unsigned raw = claim.start(threadIdx.x);
#pragma unroll
        for (int j = 0; j < R; j++) v[j] = ar.from_canonical(x[j]);
        if (!line_fwd<AR, SA, RL>(v, w, tw, 1u, u, ar, at, claim, raw)) return;
#pragma unroll
        for (int j = 0; j < R; j++) put<SHARED>(col + (long)(u * R + j) * N2, ar.to_mid_fwd(v[j]));
    } else {
        RoundTw<AR, SA, RL, SA - RL, RL> w;
        w.load(tw, 1u, u);
#pragma unroll
        for (int j = 0; j < R; j++) x[j] = get<SHARED>(col + (long)(u * R + j) * N2);
        const unsigned counted = claim.start(threadIdx.x);
#pragma unroll
        for (int j = 0; j < R; j++) v[j] = ar.from_mid(x[j]);
        line_inv<AR, SA, RL, true>(v, w, tw, 1u, u, ar, at);
        line_inv_last<AR, SA, RL>(v, x, ar);
#pragma unroll
        for (int h = 0; h < LR::GROUPS; h++)
#pragma unroll
            for (int j = 0; j < (1 << C0); j++) col[LR::pos(LR::group(u, h), j) * N2] = x[(h << C0) + j];
        claim.publish(threadIdx.x, counted);
    }
}

template <class AR, int SA, int SB, bool INVERSE, bool SHARED>
__device__ __forceinline__ void fine_row_tile(u64* limb, unsigned tile, const typename AR::TW* __restrict__ tw, const AR& ar, typename AR::V* lds,
                                              const TileClaim& claim = TileClaim()) {
    typedef FineRow<SA, SB, FINE_RL> F;
    constexpr int RL = FINE_RL, R = 1 << RL, C0 = line_first<SB, RL>(), N1 = 1 << SA;
    constexpr long N2 = 1l << SB;
    const unsigned u = threadIdx.x % F::U, rl = threadIdx.x / F::U;
    const unsigned row = tile * F::ROWS + rl, tw_off = N1 + row;
    u64* rp = limb + row * N2;
    typename AR::V* lrow = lds + rl * F::PITCH;
    auto at = [&](unsigned p) { return lrow + padded((int)p); };
    typedef LineRound<SB, RL, 0, C0> LR;
    typename AR::V v[R];
    u64 x[R];
    if constexpr (!INVERSE) {
        RoundTw<AR, SB, RL, 0, C0> w;
        w.load(tw, tw_off, u);
#pragma unroll
        for (int h = 0; h < LR::GROUPS; h++)
#pragma unroll
            for (int j = 0; j < (1 << C0); j++) x[(h << C0) + j] = get<SHARED>(rp + LR::pos(LR::group(u, h), j));
        const unsigned counted = claim.start(threadIdx.x);
#pragma unroll
        for (int j = 0; j < R; j++) v[j] = ar.from_mid(x[j]);
        line_fwd<AR, SB, RL>(v, w, tw, tw_off, u, ar, at);
#pragma unroll
        for (int j = 0; j < R; j++) x[j] = ar.to_canonical_fwd(v[j]);
        store_adjacent(rp + u * R, x);
        claim.publish(threadIdx.x, counted);
    } else {
        RoundTw<AR, SB, RL, SB - RL, RL> w;
        w.load(tw, tw_off, u);
        load_adjacent(rp + u * R, x);
        const unsigned raw = claim.start(threadIdx.x);
#pragma unroll
        for (int j = 0; j < R; j++) v[j] = ar.from_canonical(x[j]);
        if (!line_inv<AR, SB, RL, false>(v, w, tw, tw_off, u, ar, at, claim, raw)) return;
#pragma unroll
        for (int h = 0; h < LR::GROUPS; h++)
#pragma unroll
            for (int j = 0; j < (1 << C0); j++) put<SHARED>(rp + LR::pos(LR::group(u, h), j), ar.to_mid_inv(v[(h << C0) + j]));
    }
}

template <int SA, int SB> constexpr int fine_lds_words() {
    return FineStrided<SA, SB, FINE_RL>::LDS_WORDS > FineRow<SA, SB, FINE_RL>::LDS_WORDS ? FineStrided<SA, SB, FINE_RL>::LDS_WORDS : FineRow<SA, SB, FINE_RL>::LDS_WORDS;
}
template <class AR, int SA, int SB, bool INVERSE>
__global__ __launch_bounds__((FineStrided<SA, SB, FINE_RL>::THREADS)) void fine_strided_kernel(NttArgs a) {
    constexpr long N = 1l << (SA + SB);
    __shared__ typename AR::V lds[FineStrided<SA, SB, FINE_RL>::LDS_WORDS];
    int prime;
    u64* limb = limb_ptr(a, blockIdx.y, N, prime);
    const AR ar(a.primes[prime]);
    fine_strided_tile<AR, SA, SB, INVERSE, false>(limb, blockIdx.x, (const typename AR::TW*)a.tw + (long)prime * N, ar, lds);
}
template <class AR, int SA, int SB, bool INVERSE>
__global__ __launch_bounds__((FineRow<SA, SB, FINE_RL>::THREADS)) void fine_row_kernel(NttArgs a) {
    constexpr long N = 1l << (SA + SB);
    __shared__ typename AR::V lds[FineRow<SA, SB, FINE_RL>::LDS_WORDS];
    int prime;
    u64* limb = limb_ptr(a, blockIdx.y, N, prime);
    const AR ar(a.primes[prime]);
    fine_row_tile<AR, SA, SB, INVERSE, false>(limb, blockIdx.x, (const typename AR::TW*)a.tw + (long)prime * N, ar, lds);
}
// both passes in one launch of one workgroup per (limb, tile)
template <class AR, int SA, int SB, bool INVERSE>
__global__ __launch_bounds__((FineStrided<SA, SB, FINE_RL>::THREADS)) void fine_pair_kernel(NttArgs a, PairArgs p) {
    constexpr unsigned TILES = FineStrided<SA, SB, FINE_RL>::TILES;
    constexpr long N = 1l << (SA + SB);
    __shared__ typename AR::V lds[fine_lds_words<SA, SB>()];
    __shared__ unsigned go;
    unsigned limb_id, tile;
    pair_block(p, blockIdx.x, TILES, limb_id, tile);
    if (limb_id >= p.limbs) return;                                             // uniform over the workgroup
    int prime;
    u64* limb = limb_ptr(a, limb_id, N, prime);
    const AR ar(a.primes[prime]);
    const typename AR::TW* __restrict__ tw = (const typename AR::TW*)a.tw + (long)prime * N;
    pair_run<TILES>(p, limb_id, tile, &go, p.steal != 0,
                    [&](unsigned t, const TileClaim& claim) {
                        if constexpr (!INVERSE) fine_strided_tile<AR, SA, SB, false, true>(limb, t, tw, ar, lds, claim);
                        else fine_row_tile<AR, SA, SB, true, true>(limb, t, tw, ar, lds, claim);
                    },
                    [&](unsigned t, const TileClaim& out) {
                        if constexpr (!INVERSE) fine_row_tile<AR, SA, SB, false, true>(limb, t, tw, ar, lds, out);
                        else fine_strided_tile<AR, SA, SB, true, true>(limb, t, tw, ar, lds, out);
                    });
}

// whole limb: values per lane chosen so that a workgroup has at most 1024 lanes
template <int S> constexpr int whole_rl() { return S <= 13 ? 3 : 4; }
template <class AR, int S, bool INVERSE>
__global__ __launch_bounds__((FineWhole<S, whole_rl<S>()>::THREADS)) void fine_whole_kernel(NttArgs a) {
    constexpr int RL = whole_rl<S>(), R = 1 << RL, C0 = line_first<S, RL>();
    typedef FineWhole<S, RL> F;
    constexpr long N = 1l << S;
    typedef typename AR::TW TW;
    __shared__ typename AR::V lds[F::LDS_WORDS];
    int prime;
    u64* limb = limb_ptr(a, blockIdx.x, N, prime);
    const AR ar(a.primes[prime]);
    const TW* __restrict__ tw = (const TW*)a.tw + (long)prime * N;
    const unsigned u = threadIdx.x;
    auto at = [&](unsigned p) { return lds + padded((int)p); };
    typedef LineRound<S, RL, 0, C0> LR;
    typename AR::V v[R];
    u64 x[R];
    if constexpr (!INVERSE) {
        RoundTw<AR, S, RL, 0, C0> w;
        w.load(tw, 1u, u);
#pragma unroll
        for (int h = 0; h < LR::GROUPS; h++)
#pragma unroll
            for (int j = 0; j < (1 << C0); j++) x[(h << C0) + j] = limb[LR::pos(LR::group(u, h), j)];
#pragma unroll
        for (int j = 0; j < R; j++) v[j] = ar.from_canonical(x[j]);
        line_fwd<AR, S, RL>(v, w, tw, 1u, u, ar, at);
#pragma unroll
        for (int j = 0; j < R; j++) x[j] = ar.to_canonical_fwd(v[j]);
        store_adjacent(limb + u * R, x);
    } else {
        RoundTw<AR, S, RL, S - RL, RL> w;
        w.load(tw, 1u, u);
        load_adjacent(limb + u * R, x);
#pragma unroll
        for (int j = 0; j < R; j++) v[j] = ar.from_canonical(x[j]);
        line_inv<AR, S, RL, true>(v, w, tw, 1u, u, ar, at);
        line_inv_last<AR, S, RL>(v, x, ar);
#pragma unroll
        for (int h = 0; h < LR::GROUPS; h++)
#pragma unroll
            for (int j = 0; j < (1 << C0); j++) limb[LR::pos(LR::group(u, h), j)] = x[(h << C0) + j];
    }
}

// Protocol words of a paired call: a region per stream of the context, so that calls of one context on several streams (each with
// data of its own) do not count on each other's words; within a stream the calls follow one another and a call leaves its words at
// zero.  -1: no region left, or the call is being captured into a graph (its replays may run beside the stream's own calls); the
// caller then takes a form that needs no words.
constexpr int FINE_REGION = 256, FINE_REGIONS = PAIR_MAX_LIMBS / FINE_REGION;
static int pair_region(ckks_ctx* c) {
    hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(c->stream, &capturing) != hipSuccess) { (void)hipGetLastError(); return -1; }
    if (capturing != hipStreamCaptureStatusNone) return -1;
    std::lock_guard<std::mutex> lock(c->pair_streams_mutex);
    for (size_t i = 0; i < c->pair_streams.size(); i++)
        if (c->pair_streams[i] == c->stream) return (int)i;
    if (c->pair_streams.size() >= (size_t)FINE_REGIONS) return -1;
    c->pair_streams.push_back(c->stream);
    return (int)c->pair_streams.size() - 1;
}

template <class AR, int S>
static int launch_whole(ckks_ctx* c, const NttArgs& a, int limbs, bool inverse) {
    const dim3 g((unsigned)limbs), b(FineWhole<S, whole_rl<S>()>::THREADS);
    if (!inverse) hipLaunchKernelGGL((fine_whole_kernel<AR, S, false>), g, b, 0, c->stream, a);
    else hipLaunchKernelGGL((fine_whole_kernel<AR, S, true>), g, b, 0, c->stream, a);
    CKKS_HIP_TRY(hipGetLastError());
    return CKKS_OK;
}
template <class AR, int SA, int SB>
static int launch_fine(ckks_ctx* c, const NttArgs& a, int limbs, bool inverse, bool pair) {
    typedef FineStrided<SA, SB, FINE_RL> FS;
    typedef FineRow<SA, SB, FINE_RL> FR;
    if (pair) {
        const int region = limbs <= FINE_REGION ? pair_region(c) : -1;
        if (region < 0) return launch_fine<AR, SA, SB>(c, a, limbs, inverse, false);
        PairArgs p = pair_args(c, limbs);
        p.done += (size_t)region * FINE_REGION * PAIR_WORD_STRIDE;
        p.spread = 0;                                   // a limb's tiles on one XCD: spread over all of them 20.2 us against 16.0 (N = 2^15, 48 limbs)
        const dim3 g(pair_blocks(limbs, FS::TILES)), b(FS::THREADS);
        if (!inverse) hipLaunchKernelGGL((fine_pair_kernel<AR, SA, SB, false>), g, b, 0, c->stream, a, p);
        else hipLaunchKernelGGL((fine_pair_kernel<AR, SA, SB, true>), g, b, 0, c->stream, a, p);
        CKKS_HIP_TRY(hipGetLastError());
        return CKKS_OK;
    }
    const dim3 gs(FS::TILES, limbs), bs(FS::THREADS), gr(FR::TILES, limbs), br(FR::THREADS);
    if (!inverse) {
        hipLaunchKernelGGL((fine_strided_kernel<AR, SA, SB, false>), gs, bs, 0, c->stream, a);
        hipLaunchKernelGGL((fine_row_kernel<AR, SA, SB, false>), gr, br, 0, c->stream, a);
    } else {
        hipLaunchKernelGGL((fine_row_kernel<AR, SA, SB, true>), gr, br, 0, c->stream, a);
        hipLaunchKernelGGL((fine_strided_kernel<AR, SA, SB, true>), gs, bs, 0, c->stream, a);
    }
    CKKS_HIP_TRY(hipGetLastError());
    return CKKS_OK;
}

template <class AR>
static int launch(ckks_ctx* c, NttArgs a, int limbs, bool inverse, int form) {
    a.limb_base = 0;
    a.limbs_total = (unsigned)limbs;
    a.mid = nullptr;
    if (form == 1) {
        switch (c->logN) {
            case 12: return launch_whole<AR, 12>(c, a, limbs, inverse);
            case 13: return launch_whole<AR, 13>(c, a, limbs, inverse);
            case 14: return launch_whole<AR, 14>(c, a, limbs, inverse);
        }
    } else {
        switch (c->logN) {
            case 13: return launch_fine<AR, 7, 6>(c, a, limbs, inverse, form == 3);
            case 14: return launch_fine<AR, 7, 7>(c, a, limbs, inverse, form == 3);
            case 15: return launch_fine<AR, 8, 7>(c, a, limbs, inverse, form == 3);
            case 16: return launch_fine<AR, 8, 8>(c, a, limbs, inverse, form == 3);
        }
    }
    set_error("NTT: fine form outside its ring sizes");
    return CKKS_E_INVALID;
}
int launch_ntt_fine(ckks_ctx* c, const NttArgs& a, int limbs, bool inverse, int back_end, int form) {
    switch (back_end) {
        case 0: return launch<F64Arith>(c, a, limbs, inverse, form);
        case 1: return launch<F64WideArith>(c, a, limbs, inverse, form);
        case 3: return launch<PmArith>(c, a, limbs, inverse, form);
        default: return launch<IntArith>(c, a, limbs, inverse, form);
    }
}

// Workgroups of the paired kernels of the context's ring size that the chip holds at once, by back end.
template <class AR, int SA, int SB>
static unsigned fine_pair_resident(unsigned cus) {
    auto ask = [](auto kernel) {
        int n = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, kernel, FineStrided<SA, SB, FINE_RL>::THREADS, 0) != hipSuccess) { (void)hipGetLastError(); n = 1; }
        return n < 1 ? 1u : (unsigned)n;
    };
    // workgroups per compute unit: a property of the compiled kernels, asked for once
    static const unsigned fwd = ask(fine_pair_kernel<AR, SA, SB, false>), inv = ask(fine_pair_kernel<AR, SA, SB, true>);
    return (fwd < inv ? fwd : inv) * cus;
}
template <int SA, int SB>
static void fine_init(ckks_ctx* c, unsigned cus) {
    c->fine_pair_blocks[0] = fine_pair_resident<F64Arith, SA, SB>(cus);
    c->fine_pair_blocks[1] = fine_pair_resident<F64WideArith, SA, SB>(cus);
    c->fine_pair_blocks[2] = fine_pair_resident<IntArith, SA, SB>(cus);
    c->fine_pair_blocks[3] = fine_pair_resident<PmArith, SA, SB>(cus);
}
void ntt_fine_init(ckks_ctx* c) {
    const unsigned cus = (unsigned)(c->cu_count > 0 ? c->cu_count : 1);
    switch (c->logN) {
        case 13: return fine_init<7, 6>(c, cus);
        case 14: return fine_init<7, 7>(c, cus);
        case 15: return fine_init<8, 7>(c, cus);
        case 16: return fine_init<8, 8>(c, cus);
    }
}

// Which form a call of `limbs` limbs takes: 0 those of ntt.hip, 1 whole limbs in one workgroup, 2 two passes with eight values per
// lane (a setting only), 3 the same paired in one launch.
// The lines, from forward / inverse times in us of (two launches of ntt.hip, whole, paired), 36-bit primes unless said:
//   N = 2^12: whole at every size - 1 limb (7.5, 5.2), 48 (8.6 / 8.1, 5.8 / 5.2), 192 (12.7, 7.0 / 5.8), 768 (19.9, 15.6 / 11.7).
//   N = 2^13: one compute unit needs 8.2 us for a limb however few there are (11.5 in integers), so small batches are paired:
//     24 (8.9, 8.8, 7.5 / 7.1), 64 (11.1, 9.3 / 8.5, 8.5 / 7.6), 80 (12.9, 9.7 / 8.6, 10.1 / 9.1), 192 (19.5, 12.0 / 9.8, 14.0 / 11.6),
//     384 (21, 19 / 15); 60-bit: 64 (13.8, 12.3, 9.9 / 9.4), 128 (19.5, 13.5 / 12.8, 12.6 / 11.8), 160 (22.6, 14.3 / 13.1, 14.7 / 14.0).
//   N = 2^14 (a limb fills a compute unit's LDS: one round of whole limbs is 256): 64 (17.6, 15.8 / 16.9, 11.5 / 10.4), 128 (27, 18.2 / 18.0,
//     17.7 / 15.7), 160 (24, 19.1 / 18.1, 20.7 / 18.1), 256 (25.3, 22.8 / 19.2, 31), 384 (35.8, 40 / 35, 44);
//     60-bit: 160 (30, 25.6 / 24.8, 23.1 / 21.3), 192 (30, 26.7 / 25.0, 26.4 / 24.8), 256 (33.5, 29.0 / 26.9, 34).
//   N = 2^15 (no whole form): 48 (22.4, -, 16.0 / 13.9), 80 (24.4, -, 23.5 / 20.3), 96 (23.0, -, 25.2 / 22.0);
//     60-bit: 48 (27.7, -, 19.0 / 17.7), 96 (30.4, -, 26.7 / 25.7), 108 (32.9, -, 33.1).
//   N = 2^16: primes below 2^50 keep the paired kernel of ntt.hip with its 5-byte values; 60-bit primes: 8 (14.5, -, 12.8 / 12.4), 32 (23.0, -,
//     21.6 / 19.8), 48 (29.3 / 31.0, -, 29.6 / 28.1), 64 (35.6, -, 37).
// What a paired launch hands over stays in the L2 of one XCD (a limb's tiles go to one), two launches send it through the fabric.
int ntt_fine_form(const ckks_ctx* c, int limbs, int back_end) {
    const int logN = c->logN;
    if (c->ntt_fine == 4 || c->ntt_mode != 0 || c->ev_mid_armed || logN < 12) return 0;
    const bool integers = back_end >= 2;
    const bool can_pair = logN >= 13 && c->d_ntt_pair && limbs <= FINE_REGION;
    if (c->ntt_fine == 1) return logN <= 14 ? 1 : 0;
    if (c->ntt_fine == 2) return logN >= 13 ? 2 : 0;
    if (c->ntt_fine == 3) return can_pair ? 3 : 0;
    const int pair_most = logN == 13 ? (integers ? 128 : 64) : logN == 14 ? (integers ? 160 : 128) : logN == 15 ? (integers ? 96 : 80) : integers ? 40 : 0;
    const unsigned tiles = logN == 16 ? 16u : logN == 13 ? 4u : 8u;
    // paired only while the whole grid fits the chip at once: workgroups that wait for ones that cannot start yet gain nothing
    if (can_pair && limbs <= pair_most && pair_blocks(limbs, tiles) <= c->fine_pair_blocks[back_end]) return 3;
    if (logN <= 13 || (logN == 14 && limbs > 128 && limbs <= c->cu_count)) return 1;
    return 0;
}

}  // namespace ckks
