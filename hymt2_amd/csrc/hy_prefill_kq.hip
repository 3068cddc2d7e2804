// Multi-token GEMM of the Q4_K and Q6_K formats on int8 MFMA, gfx950: the contractions of a
// Q4_K_M model's prompt batches and prefill chunks.
//
// The reference multiplies (row, token) pairs block by block (src/kernels.c:808-877):
//   Q4_K: acc += y.d * (d * (float)sumi - dmin * (float)summ),  sumi = sum_j sc_j (q . y)_j over the
//         block's 8 sub-blocks of 32 (q 0..15, sc 6 bits), summ = sum_j mn_j bsum_j
//   Q6_K: acc += f16(d) * y.d * (float)tot,  tot = sum_j sc_j ((q - 32) . y)_j over 16 sub-blocks of
//         16 (q 6 bits, sc int8)
// The integers are exact in any order, so the scales move into the weight operand: each weight
// times its sub-block's scale, split into two int8 digits, is what v_mfma_i32_16x16x64_i8
// contracts, two MFMAs a K = 64 chunk, with nothing left to do per sub-block:
//   Q4_K: sc = 8 sh + sl (3 bits each): q sl and q sh are at most 105, both byte-wise products of
//         four weights by one packed 16-bit multiply a pair (no carry between bytes);
//         sumi = 8 H + L. summ comes from one v_mfma_f32_16x16x16_f16 over the block's 16 bsums
//         (|bsum| <= 2032 and mn <= 63 are exact in f16, every partial sum is an integer below 2^24).
//   Q6_K: w = sc (q - 32) (13 bits) in packed 16-bit multiply-adds, w = 256 hi + lo with lo int8.
// The fp32 terms are formed per output as the reference does and added in block order, so results
// are bit-identical to the single-token path.
//
// Layout. Tokens are the MFMA's A rows and weight rows its B columns: a lane (tl = lane % 16, kg =
// lane / 16) decodes 16-byte pieces kg of weight row tl, whose block scales it also holds, and
// receives the outputs of tokens 4 kg .. 4 kg + 3 for that row. What bounds it is the decoding: about
// 150 (Q4_K) and 270 (Q6_K) vector instructions a block step and wavefront, against 128 cycles of
// MFMA a token tile (counters at 16 tokens: vector issue 46 % of the wavefronts' cycles, MFMA 5 %). A wavefront owns one 16-row tile
// (two in pair mode: gate and up of the same rows) by NT 16-token tiles; the W wavefronts of a
// workgroup take consecutive row tiles of the same tokens, so weights go from memory to registers
// (nothing of them is shared) and the tokens' Q8_K pieces go through a double-buffered LDS stage,
// one barrier a block. KS > 1 splits K over KS sets of W wavefronts: a set keeps the fp32
// terms of its blocks in registers and they are added set after set, in block order.
#include <algorithm>

#include "hy_kernels.h"

namespace hy {

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef _Float16 v4h __attribute__((ext_vector_type(4)));
// (arrays of these stay in registers; of HIP's uint4 structs they do not)
typedef unsigned v4u __attribute__((ext_vector_type(4)));
typedef unsigned v2u __attribute__((ext_vector_type(2)));
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ uint32_t pk_mul(uint32_t a, uint32_t b) {
    return __builtin_bit_cast(uint32_t, (u16x2)(__builtin_bit_cast(u16x2, a) * __builtin_bit_cast(u16x2, b)));
}
__device__ __forceinline__ uint32_t pk_mad(uint32_t a, uint32_t b, uint32_t c) {
    return __builtin_bit_cast(
        uint32_t, (u16x2)(__builtin_bit_cast(u16x2, a) * __builtin_bit_cast(u16x2, b) + __builtin_bit_cast(u16x2, c)));
}
__device__ __forceinline__ uint32_t pair16(uint32_t v) { return v | v << 16; }

// One lane's share of one row's 256-weight block, as loaded.
template <int KIND>
struct KqSeg;
template <>
struct KqSeg<KIND_Q4K> {
    v4u hdr;   // d, dmin, the 12 scale bytes
    v4u p[2];  // bytes 64 p + 16 kg .. + 15 of qs
};
template <>
struct KqSeg<KIND_Q6K> {
    v4u ql[2], qh[2];  // ql bytes 64 h + 16 kg, qh bytes 32 h + 16 (kg & 1)
    v4u sc;            // the block's 16 scales
    uint32_t d;          // f16
};

// Lane offsets of a row's pieces; a load is the uniform address of (first row, block) plus one of them,
// so that no address arithmetic is left in the block loop.
template <int KIND>
struct KqOff;
template <>
struct KqOff<KIND_Q4K> {
    uint32_t hdr, p;
    __device__ __forceinline__ KqOff(int lrow, int nb, int kg) : hdr((uint32_t)(lrow * nb) * 144), p(hdr + 16 + 16 * kg) {}
};
template <>
struct KqOff<KIND_Q6K> {
    uint32_t l, h, s, d;
    __device__ __forceinline__ KqOff(int lrow, int nb, int kg)
        : l((uint32_t)(lrow * nb) * 128 + 16 * kg), h((uint32_t)(lrow * nb) * 64 + 16 * (kg & 1)),
          s((uint32_t)(lrow * nb) * 16), d((uint32_t)(lrow * nb) * 2) {}
};

template <class T>
__device__ __forceinline__ T kq_at(const void* base, uint32_t off) {
    return *reinterpret_cast<const T*>(static_cast<const char*>(base) + off);
}

template <int KIND>
__device__ __forceinline__ void kq_load(KqSeg<KIND>& S, const MvWeight& W, size_t blk, const KqOff<KIND>& o) {
    if constexpr (KIND == KIND_Q4K) {
        const uint8_t* b = W.w + blk * 144;
        S.hdr = kq_at<v4u>(b, o.hdr);
        S.p[0] = kq_at<v4u>(b, o.p);
        S.p[1] = kq_at<v4u>(b, o.p + 64);
    } else {
        const uint8_t *l = W.w + blk * 128, *h = W.w2 + blk * 64;
        S.ql[0] = kq_at<v4u>(l, o.l);
        S.ql[1] = kq_at<v4u>(l, o.l + 64);
        S.qh[0] = kq_at<v4u>(h, o.h);
        S.qh[1] = kq_at<v4u>(h, o.h + 32);
        S.sc = kq_at<v4u>(W.sc + blk * 16, o.s);
        S.d = kq_at<uint16_t>(W.dh + blk, o.d);
    }
}

// The four K = 64 chunks of a block. Piece of the token's natural-order qs (16 bytes each) that
// lane kg meets in chunk c. Q4_K: chunk 2 p + hi holds the low (hi = 0) or high nibbles of the
// lanes' pieces p, whose 64-weight group is 2 p + kg / 2; Q6_K: natural order.
template <int KIND>
__device__ __forceinline__ int kq_piece(int c, int kg) {
    if (KIND == KIND_Q4K) return 4 * (2 * (c >> 1) + (kg >> 1)) + 2 * (c & 1) + (kg & 1);
    return 4 * c + kg;
}

// Per block and lane: what the chunks' decoding and the terms need.
template <int KIND>
struct KqBlock;
template <>
struct KqBlock<KIND_Q4K> {
    uint32_t s[2];  // scales of the lane's sub-blocks, bytes (low nibbles, high nibbles) of piece p
    v4h mn;         // f16 mins of k = 4 kg .. 4 kg + 3 of the 16 bsums: mn[2 kg] twice, mn[2 kg + 1] twice
    float d, dmin;
};
template <>
struct KqBlock<KIND_Q6K> {
    float d;
};

template <int KIND>
__device__ __forceinline__ void kq_block(KqBlock<KIND>& B, const KqSeg<KIND>& S, int kg) {
    if constexpr (KIND == KIND_Q4K) {
        // scale and min j (src/kernels.c:839-842), the bytes of j and j + 1 together: j = 2 (kg / 2)
        // and 4 + that for the scales, j = 2 kg for the mins
        const int sh = 16 * (kg >> 1), mh = 16 * (kg & 1);
        const uint32_t y = S.hdr.y >> sh, w = S.hdr.w >> sh;
        B.s[0] = y & 0x3f3fu;
        B.s[1] = (w & 0x0f0fu) | ((y >> 2) & 0x3030u);
        const uint32_t z = S.hdr.z >> mh, wm = S.hdr.w >> (mh + 4);
        const uint32_t m = kg < 2 ? z & 0x3f3fu : (wm & 0x0f0fu) | ((z >> 2) & 0x3030u);
        const _Float16 m0 = (_Float16)(unsigned short)(m & 0xffu), m1 = (_Float16)(unsigned short)((m >> 8) & 0xffu);
        B.mn = v4h{m0, m0, m1, m1};
        B.d = hy_f16((uint16_t)(S.hdr.x & 0xffffu));
        B.dmin = hy_f16((uint16_t)(S.hdr.x >> 16));
    } else {
        B.d = hy_f16((uint16_t)S.d);
    }
}

// The two int8 digits of the scaled weights of chunk c: high part times HB plus low part.
template <int KIND>
struct KqDigits {
    static constexpr int SHIFT = KIND == KIND_Q4K ? 3 : 8;  // w = (hi << SHIFT) + lo
};
template <int KIND>
__device__ __forceinline__ void kq_chunk(const KqSeg<KIND>& S, const KqBlock<KIND>& B, int c, int kg, v4i& lo, v4i& hi) {
    if constexpr (KIND == KIND_Q4K) {
        const v4u p = S.p[c >> 1];
        const uint32_t s = (B.s[c >> 1] >> (8 * (c & 1))) & 63u;
        const uint32_t sl = pair16(s & 7u), sh = pair16(s >> 3);
        const uint32_t w[4] = {p.x, p.y, p.z, p.w};
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t q = (w[i] >> (4 * (c & 1))) & 0x0f0f0f0fu;
            lo[i] = (int)pk_mul(q, sl);
            hi[i] = (int)pk_mul(q, sh);
        }
    } else {
        const v4u l4 = S.ql[c >> 1], h4 = S.qh[c >> 1];
        const uint32_t wl[4] = {l4.x, l4.y, l4.z, l4.w}, wh[4] = {h4.x, h4.y, h4.z, h4.w};
        const uint32_t scw[4] = {S.sc.x, S.sc.y, S.sc.z, S.sc.w};
        const int sc = (int)(scw[c] << (24 - 8 * kg)) >> 24;  // scale 4 c + kg
        const uint32_t scp = pair16((uint32_t)sc & 0xffffu);
        const uint32_t cst = pair16((uint32_t)(128 - 32 * sc) & 0xffffu);
        const int qs = 2 * (kg >> 1);  // the lane's 2-bit field of qh for low nibbles (high: 4 further)
#pragma unroll
        for (int i = 0; i < 4; i++) {
            // the 6-bit value's nibble and, moved to bits 4 and 5, its qh field (bits 6 and 7: others')
            const uint32_t x = (c & 1) == 0 ? wh[i] << (4 - qs) : wh[i] >> qs, y = (c & 1) == 0 ? wl[i] : wl[i] >> 4;
            const uint32_t u = (y & 0x0f0f0f0fu) | (x & 0xf0f0f0f0u);
            // sc (q - 32) + 128 of weights 0, 2 and 1, 3
            const uint32_t pe = pk_mad(u & 0x003f003fu, scp, cst), po = pk_mad((u >> 8) & 0x003f003fu, scp, cst);
            hi[i] = (int)__builtin_amdgcn_perm(po, pe, 0x07030501u);
            lo[i] = (int)(__builtin_amdgcn_perm(po, pe, 0x06020400u) ^ 0x80808080u);
        }
    }
}

// One 256-element block of the workgroup's tokens in LDS: piece c of token t's qs at slot
// 16 t + (c ^ (t & 15)), so that the 16 tokens of an A-fragment read hit 16 bank groups; the bsums
// as f16; the Q8_K scales.
template <int T>
struct KqStage {
    alignas(16) uint8_t q[T * 256];
    alignas(16) _Float16 bs[T * 16];
    alignas(16) float d[T];
};

// A thread's share of one block of T tokens (THR threads), between its global loads and LDS stores.
// Threads past a field's pieces repeat one (the same value to the same place): no branch splits
// the loads, which the compiler would otherwise move behind it.
template <int T, int THR, bool BS>
struct KqTok {
    static constexpr int QN = (T * 16 + THR - 1) / THR, BN = BS ? (T * 4 + THR - 1) / THR : 1;
    v4u q[QN];
    v2u b[BN];
    float d;
};

// The thread's pieces' offsets from the first token's block (tokens past the last repeat it).
template <int T, int THR, bool BS>
struct KqTokOff {
    uint32_t q[KqTok<T, THR, BS>::QN], b[KqTok<T, THR, BS>::BN], d;
    __device__ __forceinline__ KqTokOff(int nb, int left, int th) {
        auto tok = [&](int t) { return (uint32_t)(min(t, left - 1) * nb) * (uint32_t)sizeof(HyQ8K); };
#pragma unroll
        for (int i = 0; i < KqTok<T, THR, BS>::QN; i++) {
            const int f = (th + THR * i) % (T * 16);
            q[i] = tok(f / 16) + offsetof(HyQ8K, qs) + 16 * (f % 16);
        }
#pragma unroll
        for (int i = 0; i < KqTok<T, THR, BS>::BN; i++) {
            const int f = (th + THR * i) % (T * 4);
            b[i] = tok(f / 4) + offsetof(HyQ8K, bsums) + 8 * (f % 4);
        }
        d = tok(th % T) + offsetof(HyQ8K, d);
    }
};

template <int T, int THR, bool BS>
__device__ __forceinline__ void kq_tok_load(KqTok<T, THR, BS>& R, const HyQ8K* blk, const KqTokOff<T, THR, BS>& o) {
#pragma unroll
    for (int i = 0; i < R.QN; i++) R.q[i] = kq_at<v4u>(blk, o.q[i]);
    if constexpr (BS) {
#pragma unroll
        for (int i = 0; i < R.BN; i++) R.b[i] = kq_at<v2u>(blk, o.b[i]);
    }
    R.d = kq_at<float>(blk, o.d);
}

template <int T, int THR, bool BS>
__device__ __forceinline__ void kq_tok_store(const KqTok<T, THR, BS>& R, KqStage<T>& S, int th) {
#pragma unroll
    for (int i = 0; i < R.QN; i++) {
        const int f = (th + THR * i) % (T * 16), t = f / 16, c = f % 16;
        *reinterpret_cast<v4u*>(S.q + (16 * t + (c ^ (t & 15))) * 16) = R.q[i];
    }
    if constexpr (BS) {
#pragma unroll
        for (int i = 0; i < R.BN; i++) {
            const int f = (th + THR * i) % (T * 4);
            const v4h v = {(_Float16)(short)(R.b[i].x & 0xffffu), (_Float16)(short)(R.b[i].x >> 16),
                           (_Float16)(short)(R.b[i].y & 0xffffu), (_Float16)(short)(R.b[i].y >> 16)};
            *reinterpret_cast<v4h*>(S.bs + 4 * f) = v;
        }
    }
    S.d[th % T] = R.d;
}

template <int NT, int W, int KS>
struct KqLds {
    union {
        KqStage<16 * NT> st[2][KS];
        float xch[KS > 1 ? W * 64 * 2 * NT * 4 : 1];  // sums handed from one K set to the next
    };
    uint64_t etab[32];  // expf table of the SwiGLU epilogue
};

// The fp32 terms of one block for the wavefront's MT x NT tiles.
template <int KIND, int MT, int NT>
__device__ __forceinline__ void kq_step(const KqSeg<KIND> (&seg)[MT], const KqStage<16 * NT>& S, int tl, int kg,
                                        float (&term)[MT][NT][4]) {
    KqBlock<KIND> B[MT];
    v4i H[MT][NT], Lo[MT][NT];
#pragma unroll
    for (int m = 0; m < MT; m++) {
        kq_block<KIND>(B[m], seg[m], kg);
#pragma unroll
        for (int n = 0; n < NT; n++) H[m][n] = Lo[m][n] = v4i{0, 0, 0, 0};
    }
#pragma unroll
    for (int c = 0; c < 4; c++) {
        v4i a[NT];
        const int pc = kq_piece<KIND>(c, kg);
#pragma unroll
        for (int n = 0; n < NT; n++)
            a[n] = *reinterpret_cast<const v4i*>(S.q + (16 * (16 * n + tl) + (pc ^ tl)) * 16);
#pragma unroll
        for (int m = 0; m < MT; m++) {
            v4i lo, hi;
            kq_chunk<KIND>(seg[m], B[m], c, kg, lo, hi);
#pragma unroll
            for (int n = 0; n < NT; n++) {
                H[m][n] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[n], hi, H[m][n], 0, 0, 0);
                Lo[m][n] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[n], lo, Lo[m][n], 0, 0, 0);
            }
        }
    }
#pragma unroll
    for (int n = 0; n < NT; n++) {
        const float4 y4 = *reinterpret_cast<const float4*>(&S.d[16 * n + 4 * kg]);
        const float yd[4] = {y4.x, y4.y, y4.z, y4.w};
        v4h bs;
        if constexpr (KIND == KIND_Q4K) bs = *reinterpret_cast<const v4h*>(&S.bs[16 * (16 * n + tl) + 4 * kg]);
#pragma unroll
        for (int m = 0; m < MT; m++) {
            if constexpr (KIND == KIND_Q4K) {
                const v4f sm = __builtin_amdgcn_mfma_f32_16x16x16f16(bs, B[m].mn, v4f{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
                for (int r = 0; r < 4; r++)  // src/kernels.c:875
                    term[m][n][r] = yd[r] * (B[m].d * (float)((H[m][n][r] << 3) + Lo[m][n][r]) - B[m].dmin * sm[r]);
            } else {
#pragma unroll
                for (int r = 0; r < 4; r++)  // src/kernels.c:833
                    term[m][n][r] = B[m].d * yd[r] * (float)((H[m][n][r] << 8) + Lo[m][n][r]);
            }
        }
    }
}

// One workgroup's tile of job J (KIND its weights' kind; UP: a pair's up weights): W row tiles
// from row0 by tokens t0 .. t0 + 16 NT. NBH: blocks a K set holds (KS > 1; past the last: unused).
template <int KIND, int NT, int W, int KS, int NBH, bool PAIR>
__device__ __forceinline__ void kq_tile(const GemmJob& J, const MvWeight& UP, int nb, int row0, int t0, KqLds<NT, W, KS>& S) {
    constexpr int MT = PAIR ? 2 : 1, T = 16 * NT, THR = 64 * W;
    constexpr bool BS = KIND == KIND_Q4K;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), set = KS > 1 ? wave / W : 0, wr = KS > 1 ? wave % W : wave;
    const int th = KS > 1 ? tid - set * THR : tid;
    const int tl = lane & 15, kg = lane >> 4;
    const int nt = J.nt, n = J.W.n;
    const int row = row0 + 16 * wr + tl;  // this lane's weight row
    const KqOff<KIND> wo(min(row, n - 1) - row0, nb, kg);
    const KqTokOff<T, THR, BS> to(nb, nt - t0, th);
    const HyQ8K* const act = J.act + (size_t)t0 * nb;
    const int nbs = KS > 1 ? NBH : nb, b0 = set * nbs;  // blocks of this set
    auto blk = [&](int b) { return min(b0 + min(b, nbs - 1), nb - 1); };

    // Loads run about two blocks ahead (a block step is shorter than a load's round trip): weights in
    // two register sets, refilled behind their last use; tokens in two sets on their way to the
    // stage that the block before last has left. Waits are in issue order, so the token loads,
    // waited for a step before their weights, need the longer lead.
    KqTok<T, THR, BS> tk[2];
    KqSeg<KIND> seg[2][MT];
    auto load_tok = [&](int b, KqTok<T, THR, BS>& k) __attribute__((always_inline)) {
        kq_tok_load<T, THR, BS>(k, act + blk(b), to);
    };
    auto load_w = [&](int b, KqSeg<KIND> (&w)[MT]) __attribute__((always_inline)) {
#pragma unroll
        for (int m = 0; m < MT; m++) kq_load<KIND>(w[m], m ? UP : J.W, (size_t)row0 * nb + blk(b), wo);
    };
    load_tok(0, tk[0]);
    load_w(0, seg[0]);
    load_tok(1, tk[1]);
    load_w(1, seg[1]);
    __builtin_amdgcn_sched_barrier(0);
    kq_tok_store<T, THR, BS>(tk[0], S.st[0][set], th);
    load_tok(2, tk[0]);

    float acc[MT][NT][4];
#pragma unroll
    for (int m = 0; m < MT; m++)
#pragma unroll
        for (int k = 0; k < NT; k++)
#pragma unroll
            for (int r = 0; r < 4; r++) acc[m][k][r] = 0.f;
    auto add = [&](const float (&t)[MT][NT][4]) __attribute__((always_inline)) {
#pragma unroll
        for (int m = 0; m < MT; m++)
#pragma unroll
            for (int k = 0; k < NT; k++)
#pragma unroll
                for (int r = 0; r < 4; r++) acc[m][k][r] += t[m][k][r];
    };
    // block b, its weights in w; k holds block b + 1's tokens
    auto step = [&](int b, KqSeg<KIND> (&w)[MT], KqTok<T, THR, BS>& k, float (&t)[MT][NT][4]) __attribute__((always_inline)) {
        hy_lds_barrier();  // (loads stay in flight) block b is in its stage, block b - 1's has been read
        kq_tok_store<T, THR, BS>(k, S.st[(b + 1) & 1][set], th);
        load_tok(b + 3, k);
        __builtin_amdgcn_sched_barrier(0);  // the loads issue here, not next to their use
        kq_step<KIND, MT, NT>(w, S.st[b & 1][set], tl, kg, t);
        load_w(b + 2, w);
        __builtin_amdgcn_sched_barrier(0);
    };
    if constexpr (KS == 1) {
        float t[MT][NT][4];
        int b = 0;
        for (; b + 2 <= nb; b += 2) {
            step(b, seg[0], tk[1], t);
            add(t);
            step(b + 1, seg[1], tk[0], t);
            add(t);
        }
        if (b < nb) {
            step(b, seg[0], tk[1], t);
            add(t);
        }
    } else {
        float tm[NBH][MT][NT][4];
#pragma unroll
        for (int b = 0; b < NBH; b++) step(b, seg[b & 1], tk[(b + 1) & 1], tm[b]);
        // the sets' terms one set after another (through LDS that held the token stages)
        float4* const xv = reinterpret_cast<float4*>(S.xch) + (size_t)(wr * 64 + lane) * (MT * NT);
#pragma unroll
        for (int s = 0; s < KS; s++) {
            __syncthreads();
            if (set != s) continue;
#pragma unroll
            for (int m = 0; m < MT; m++)
#pragma unroll
                for (int k = 0; k < NT; k++)
                    if (s > 0) {
                        const float4 p = xv[m * NT + k];
                        acc[m][k][0] = p.x, acc[m][k][1] = p.y, acc[m][k][2] = p.z, acc[m][k][3] = p.w;
                    }
#pragma unroll
            for (int b = 0; b < NBH; b++)
                if (b0 + b < nb) add(tm[b]);
            if (s + 1 < KS)
#pragma unroll
                for (int m = 0; m < MT; m++)
#pragma unroll
                    for (int k = 0; k < NT; k++)
                        xv[m * NT + k] = make_float4(acc[m][k][0], acc[m][k][1], acc[m][k][2], acc[m][k][3]);
        }
        if (set != KS - 1) return;
    }

    if (row >= n) return;
    float* const out = J.out;
    const int ldo = J.ldo;
#pragma unroll
    for (int k = 0; k < NT; k++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int t = t0 + 16 * k + 4 * kg + r;
            if (t >= nt) continue;
            float* o = out + (size_t)t * ldo + row;
            if (PAIR) {
                const float g = acc[0][k][r];
                *o = g / (1.0f + hy_expf_tab(-g, S.etab)) * acc[MT - 1][k][r];  // SwiGLU, src/model.c:873-876
            } else {
                *o = J.epi == EPI_ADD ? *o + acc[0][k][r] : acc[0][k][r];
            }
        }
}

// Q: the launch may hold Q4_K (bit 0) and Q6_K (bit 1) jobs.
template <int Q, int NJ, int NT, int W, int KS, int NBH, bool PAIR>
__global__ __launch_bounds__(64 * W * KS) void k_gemm_kq(GemmLaunchT<NJ> L) {
    __shared__ KqLds<NT, W, KS> S;
    GemmJob J;
    MvWeight UP{};
    int begin, nb;
    const int wg = blockIdx.x;
    gemm_job<false, PAIR, NJ>(L, wg, J, UP, begin, nb);
    if (PAIR && threadIdx.x < 32) S.etab[threadIdx.x] = hy_exp_tab_entry(threadIdx.x);  // read after the block barriers
    const int row0 = (wg - begin) * 16 * W, t0 = (int)blockIdx.y * 16 * NT;
    if (t0 >= J.nt) return;  // a shorter chunk of a pipelined launch (uniform)
    if (Q == 1 || (Q == 3 && J.W.kind == KIND_Q4K)) kq_tile<KIND_Q4K, NT, W, KS, NBH, PAIR>(J, UP, nb, row0, t0, S);
    else kq_tile<KIND_Q6K, NT, W, KS, NBH, PAIR>(J, UP, nb, row0, t0, S);
}

template <int Q, int NJ, int NT, int W, int KS, int NBH, bool PAIR>
hipError_t kq_go(GemmLaunchT<NJ>& L, hipStream_t s) {
    const int tiles = gemm_tiles(L, 16 * W);
    k_gemm_kq<Q, NJ, NT, W, KS, NBH, PAIR><<<dim3(tiles, (L.nt + 16 * NT - 1) / (16 * NT)), 64 * W * KS, 0, s>>>(L);
    return hipGetLastError();
}

// K over four sets of W wavefronts, for K up to 8192 (nb <= 32).
template <int Q, int NJ, int NT, int W, bool PAIR>
hipError_t kq_split(GemmLaunchT<NJ>& L, hipStream_t s) {
    if (L.nb <= 8) return kq_go<Q, NJ, NT, W, 4, 2, PAIR>(L, s);
    if (L.nb <= 16) return kq_go<Q, NJ, NT, W, 4, 4, PAIR>(L, s);
    if (L.nb <= 24) return kq_go<Q, NJ, NT, W, 4, 6, PAIR>(L, s);
    return kq_go<Q, NJ, NT, W, 4, 8, PAIR>(L, s);
}

// The split of a launch, by token tiles and K. A block step costs a wavefront its weights' decoding
// (about 0.8 us of issue for Q6_K and 0.45 for Q4_K) and 0.1-0.2 us a token tile, however many
// wavefronts run, so few tokens want K split over wavefronts (fewer steps each) and many want
// several token tiles a wavefront (one decoding for them). Measured at the 1.8B shapes, us a launch
// in the model (the general matvec's in groups of 16 tokens in brackets):
//   16 tokens: gate/up 12.0 split, 12.2 whole (38); down 12.7 split, 27.8 whole (23.6)
//   48 tokens: gate/up 19.0 split, 21.0 whole; down 15.7 split in 2 token tiles, 18.8 in 1
//   72 tokens: gate/up 21.6 in 1 token tile, 23.3 in 4; down 18.7 in 2 rows' tiles, 20.5 in 1
//   128 tokens: gate/up 23.3 in 4 token tiles, 25.5 in 2, 32 in 1 or split (304); qkv 12.1 in 2,
//   13.3 split, 15.8 in 1 (108); down 20.9 in 2 x 2 tiles split, 24.2 in 1 x 2, 30 whole (189);
//   alone: 512 rows of Q4_K 5.1 split, 7.4 whole, of Q6_K 5.9 and 9.8 (2048 rows of Q4_K 10.0 and 7.7);
//   6144 rows of Q4_K 12.7 in 4 token tiles and K halves, 13.7 with K whole
// Single contractions of 12-32 blocks are split, in the form with the fewest tokens and rows a
// workgroup whose workgroups the CUs take at once (256 of the 256- and 512-thread ones run side by
// side; more take turns). 2048 x 6144 alone, Q4_K / Q6_K: 32 tokens 8.1 / 10.3 in 1 token tile (256
// workgroups), 10.8 / 12.6 in 2 (128); 48 tokens 12.2 / 16.0 in 1 (384), 11.3 / 12.7 in 2 (256); 64
// tokens 12.2 / 16.3 in 1 (512), 11.3 / 12.9 in 2 (256), 13.1 / 16.8 in 2 x 2 (128); 80 tokens 16.2 /
// 18.8 in 2 (384), 13.3 / 16.6 in 2 x 2 (192). 2560 x 6912 at 48 tokens: 18.2 / 21.3 in 2 (320), 14.2 /
// 18.1 in 2 x 2 (160); 4112 x 3840, where no form fits at once, 16.1 / 18.2 in 2 (514), 16.4 / 20.0 in
// 2 x 2 (258). With fewer blocks the steps are few and 384 workgroups of 1 token tile are as
// fast: 2048 x 2048 at 48 tokens 6.8 / 8.1 in 1, 7.0 / 7.5 in 2, 7.9 / 11.0 with K whole.
template <int Q, int NJ, bool PAIR>
hipError_t kq_shape(GemmLaunchT<NJ>& L, hipStream_t s) {
    int rows = 0;
    for (int q = 0; q < L.njobs; q++)
        if (!PAIR || q % 2 == 0) rows += L.job[q].W.n;
    const int tt = (L.nt + 15) / 16;
    if constexpr (NJ == kGemmPipeJobs) {
        // several chunks: K whole; 4 token tiles a wavefront once their workgroups (64 rows by 64
        // tokens) fill the chip, twice over for pairs. Two chunks of 128: pairs 37.8 us in 2 token
        // tiles, 43.6 in 4; down 32.1 and 43.0. Eight: pairs 151 and 138, down 109 and 76, qkv 55 and 39
        const int wgs = (rows + 63) / 64 * ((tt + 3) / 4);
        if (tt >= 3 && wgs >= (PAIR ? 512 : 256)) return kq_go<Q, NJ, 4, 4, 1, 1, PAIR>(L, s);
        return tt > 1 ? kq_go<Q, NJ, 2, 4, 1, 1, PAIR>(L, s) : kq_go<Q, NJ, 1, 4, 1, 1, PAIR>(L, s);
    }
    const int rt = (rows + 15) / 16, tiles = rt * tt;
    if (L.nb <= 32 && (tt == 1 || (PAIR && tt <= 3 && L.nb <= 8) || (!PAIR && tiles <= (L.nb < 12 ? 384 : 256))))
        return kq_split<Q, NJ, 1, 1, PAIR>(L, s);
    if constexpr (!PAIR)
        if (L.nb <= 32 && L.nb >= 12) {
            const int t2 = (tt + 1) / 2;
            const bool one_row = rt * t2 <= 256 || (tt <= 3 && (rt + 1) / 2 * t2 > 256);
            return one_row ? kq_split<Q, NJ, 2, 1, false>(L, s) : kq_split<Q, NJ, 2, 2, false>(L, s);
        }
    if constexpr (!PAIR)
        if (tt >= 6 && rows >= 4096 && L.nb <= 8) return kq_go<Q, NJ, 4, 4, 2, 4, false>(L, s);
    if (tt >= 6 && rows >= 4096) return kq_go<Q, NJ, 4, 4, 1, 1, PAIR>(L, s);
    if (tt >= 6 && rows > 2048) return kq_go<Q, NJ, 2, 4, 1, 1, PAIR>(L, s);
    return kq_go<Q, NJ, 1, 4, 1, 1, PAIR>(L, s);
}

// Checks the jobs and completes the launch, as the panel GEMM's gemm_prepare does.
template <int NJ>
hipError_t kq_dispatch(GemmLaunchT<NJ>& L, hipStream_t s) {
    if (L.njobs < 1 || L.njobs > NJ || (L.pair && L.njobs % 2)) return hipErrorInvalidValue;
    const int K = L.job[0].W.k;
    if (K % 256) return hipErrorNotSupported;
    int ntmax = 0, kinds = 0;
    for (int q = 0; q < L.njobs; q++) {
        GemmJob& J = L.job[q];
        const MvWeight& W = J.W;
        if ((W.kind != KIND_Q4K && W.kind != KIND_Q6K) || W.k != K || W.nb != K / 256 || W.n < 1 || !J.out)
            return hipErrorNotSupported;
        kinds |= W.kind == KIND_Q4K ? 1 : 2;
        if (!J.act) {
            J.act = L.act;
            J.nt = L.nt;
        }
        if (!J.act || J.nt < 1) return hipErrorInvalidValue;
        if (L.pair && q % 2) {
            const GemmJob& G = L.job[q - 1];
            if (W.n != G.W.n || W.kind != G.W.kind || J.act != G.act || J.nt != G.nt) return hipErrorNotSupported;
        }
        ntmax = std::max(ntmax, J.nt);
    }
    L.nt = ntmax;
    L.nb = K / 256;
    if (L.pair) return kinds == 1 ? kq_shape<1, NJ, true>(L, s) : kinds == 2 ? kq_shape<2, NJ, true>(L, s) : hipErrorNotSupported;
    return kinds == 1 ? kq_shape<1, NJ, false>(L, s) : kinds == 2 ? kq_shape<2, NJ, false>(L, s) : kq_shape<3, NJ, false>(L, s);
}

}  // namespace

hipError_t launch_gemm_kq(GemmLaunch& L, hipStream_t s) { return kq_dispatch(L, s); }
hipError_t launch_gemm_kq(GemmPipeLaunch& L, hipStream_t s) { return kq_dispatch(L, s); }

}  // namespace hy
