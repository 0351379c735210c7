// Flash attention forward with a per-head pair bias and a per-row key mask, for gfx950.
// Replaces VoltaMma (cuda/volta_mma_attn.cu:70-351) and VoltaWmma (cuda/volta_wmma_attn.cu:
// 47-311) with one kernel for f16 and bf16 on MFMA 16x16x32 with float32 accumulation.
//
// Work split: a block of 4 waves owns (query tile of 64*QT rows, head h, row n), QT chosen by
// fwd_small_blocks; each wave owns 16*QT queries and streams the keys in tiles of 64 through
// double-buffered LDS: tile kt+1 is fetched with direct global->LDS loads (K, V and the bias
// rows) while tile kt is computed, so each tile costs one barrier. Which tiles contain an absent
// key is worked out once per block from the mask row; the others skip the mask entirely.
//
// Any even Sk, and any odd one (by query parity, the ODD form below), loads its bias through LDS.
// Reading bias and mask element by element, as a ragged Sk once did, left the kernel waiting on
// sixteen 2-byte loads per lane and tile: triangle attention of 757 residues (4 heads x 32)
// 2395 -> 529 us, 1024 sequences of 300 residues (8 heads x 8) 965 -> 255 us, 203 residues
// 68 -> 23 us. That path remains for what the direct loads cannot take (fwd_form).
//
// A block runs only 5 to 16 key tiles, so what it does before and after them counts: of 22600
// cycles at 384 residues, 4600 passed before the first tile was there (2500 before its loads went
// out) and 1100 after the last. The work item comes from prepared multipliers, the arguments in
// one round of scalar loads, the mask, Q and tile loads carry no branch (a row or key that does
// not exist reads zero), and the presence words wait for the mask bytes alone: D = 32, 300
// residues 47.2 -> 45.1 us, 384 72.2 -> 69.4, 757 537 -> 515; D = 16, 300 40.5 -> 36.9;
// D = 64, 300 91.3 -> 85.5.
//
// What the fast forms cannot hold -- -inf in the bias, float16 queries whose every logit lies near
// the type's lowest value -- is found from a block's sums and maxima after its last tile, and the
// block's keys are run again in the plain form (the end of the kernel).
//
// Per 64-key tile and 16-query sub-tile a wave computes S^T = K . Q^T with the keys of each
// 32-key chunk permuted so that lane l's accumulator holds keys 8*(l/16)+0..7 of the chunk for
// query l%16. Those eight values are exactly the B operand of O^T = V^T . P^T for that chunk, so
// P never leaves registers; V^T comes from LDS with ds_read_b64_tr_b16 (two 4x16 transposed
// reads per operand). O^T accumulates four consecutive head dims per lane, stored as 8 bytes.
//
// Numerics (volta_mma_attn.cu:137,174-272): logit = scale*(q.k) + bias in float32; a key with
// kmask == 0 gets the logit -1e9 (the float32 value of the caller's additive 1e9*(mask-1)), a
// key past Sk gets -inf; online softmax in the exp2 domain, whose running max moves only when a
// tile's max exceeds it by more than 2^8 in P (so P <= 256, and O and l are rescaled on few
// tiles); P rounded to the input type for the P.V product (as the reference rounds it to f16,
// :221: the relative rounding is the same at any magnitude); O = acc / max(l, 1e-30) (:265).
// A row whose keys are all masked gets the logit 0 for them instead: its softmax is the same
// (uniform over the Sk keys), but float32 cannot subtract a running max of -1e9 exactly (its
// rounding unit there is 128), which would scale P by up to 2^64.
// lse = m + log(l) (natural log) is written when requested, for the backward pass; for an
// all-masked row it is therefore ln(Sk), relative to the masked logit. Present-key logits are
// expected above -5e8 (half the masked logit, where the running max starts): a row whose
// present keys all lie below it has no weight, O = 0 and lse = +inf (zero gradients).
#include "attention_common.hpp"

#include <type_traits>

namespace clk {
namespace {

constexpr float kRescaleSlack = 8.f;  // log2 of the largest P before the running max moves
constexpr int kGateChannels = 128;    // gate channels (wg rows) per K/V buffer in the epilogue
constexpr int kPresWords = 256;       // most key tiles of the bias-patching forward (LDS words)
constexpr float kLn2 = 0.69314718055994531f;

// Cross-group max of two values at once (lanes l, l^16, l^32, l^48 share a query): the halves
// of a and b meet in one register, so the three lane swaps serve both.
__device__ __forceinline__ void xgroup_max2(float& a, float& b) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false,
                                                    false);
    // lanes 0..31: a's lanes l and l+32; lanes 32..63: b's lanes l-32 and l
    float c = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
    const auto t = __builtin_amdgcn_permlane16_swap(__float_as_uint(c), __float_as_uint(c), false,
                                                    false);
    c = fmaxf(__uint_as_float(t[0]), __uint_as_float(t[1]));
    const auto u = __builtin_amdgcn_permlane32_swap(__float_as_uint(c), __float_as_uint(c), false,
                                                    false);
    a = __uint_as_float(u[0]);
    b = __uint_as_float(u[1]);
}

// Per-tile "some key absent or past Sk" flags of one mask row, as bits of a 64-bit word (tiles of
// 64 keys; tiles past the 64th always take the checked path), worked out by each wave on its
// own with ballots -- no LDS and no block barrier. Also returns the row's masked logit.
struct RowFlags {
    uint64_t bits;
    float masked_logit;
};
__device__ __forceinline__ RowFlags row_flags(const uint8_t* mrow, int Sk) {
    const int lane = threadIdx.x & 63;
    const int ntiles = (Sk + 63) / 64;
    // The ragged last tile (tiles from the 64th on are always checked: no bit for them).
    uint64_t bits = (Sk % 64 && ntiles <= 64) ? 1ull << (ntiles - 1) : 0ull;
    bool any_present = false;
    if (mrow) {
        for (int base = 0; base < Sk; base += 512) {
            const int k = base + 8 * lane;
            bool absent = false, present = false;
#pragma unroll
            for (int j = 0; j < 8; ++j)
                if (k + j < Sk) {
                    const bool p = mrow[k + j] != 0;
                    present |= p;
                    absent |= !p;
                }
            const uint64_t ab = __ballot(absent);
            any_present |= __ballot(present) != 0ull;
#pragma unroll
            for (int t = 0; t < 8; ++t)
                if (base / 64 + t < 64 && ((ab >> (8 * t)) & 0xffull)) bits |= 1ull << (base / 64 + t);
        }
    }
    return {bits, (mrow && !any_present) ? 0.f : kMaskedLogit};
}

// Per-lane prefetch state of one key tile of the element-wise path: the mask bytes of keys
// k0 + 32c + 8g + 0..7 (c = 0, 1) and the bias of those keys for each of the lane's query rows.
template <typename TR, int QT>
struct TilePrefetch {
    u32x2 mask[2];
    u32x4 bias[QT][2];
    __device__ __forceinline__ void load(const typename TR::elem* const* brow,
                                         const uint8_t* mrow, int k0, int g, int Sk) {
        using E = typename TR::elem;
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            const int kk = k0 + 32 * c + 8 * g;
            uint8_t m[8];
#pragma unroll
            for (int j = 0; j < 8; ++j)
                m[j] = kk + j < Sk ? (mrow ? mrow[kk + j] : uint8_t(1)) : uint8_t(0);
            __builtin_memcpy(&mask[c], m, 8);
#pragma unroll
            for (int qt = 0; qt < QT; ++qt) {
                E e[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) e[j] = kk + j < Sk ? brow[qt][kk + j] : E(0.f);
                __builtin_memcpy(&bias[qt][c], e, 16);
            }
        }
    }
    // Bit j set when key k0 + 32c + 8g + j is present.
    __device__ __forceinline__ unsigned valid(int c) const {
        unsigned bits = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            bits |= (((mask[c][0] >> (8 * j)) & 0xffu) != 0u ? 1u : 0u) << j;
            bits |= (((mask[c][1] >> (8 * j)) & 0xffu) != 0u ? 1u : 0u) << (4 + j);
        }
        return bits;
    }
};

// Operands of the output gate fused into the forward's epilogue:
//   gated[n, s, h*D + d] = O[n, h, s, d] * sigmoid(x[n, s, :] . wg[:, h*D + d] + bg[h*D + d])
// with x [N, Sq, C], wg [C, HD] row-major, bg [HD], gated [N, Sq, HD], HD = H*D, C % 32 == 0.
template <typename E>
struct GateArgs {
    const E* x;
    const E* wg;
    const E* bg;
    E* gated;
    int C, HD;
};

// A block's work item a * outer.d + b * inner.d + c from its index, the divisors prepared at
// launch: (a, b, c) are (row, head, query tile), or with grp > 0 (head, group of rows, place in it).
struct FwdItems {
    FastDiv outer, inner;     // items of one a, of one b
    FastDiv rows, last_rows;  // grp > 0: rows of a group, of the last group
    int grp, nrows;
};

// ODD (VEC, not BM): Sk is odd. The direct-to-LDS loads of the bias need 4-byte aligned addresses,
// and every other bias row starts half a dword off. A block then owns queries of one parity
// (query q0 + 2i for its i-th row), whose bias rows are all aligned or all off by one element;
// in the second case its key tiles start one key early (tile kt: keys 64kt - 1 ...), which
// aligns every load, and key -1 is an absent key. So the loop is the even one, with no shifting
// of bias pieces.
template <typename TR, int D, int QT, bool VEC, bool GATE, bool BM, bool NSHD, bool ODD>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(D <= 32 && VEC ? 3 : 1))) void attn_fwd_kernel(
    const typename TR::elem* __restrict__ q, const typename TR::elem* __restrict__ k,
    const typename TR::elem* __restrict__ v, const typename TR::elem* __restrict__ bias,
    const uint8_t* __restrict__ kmask, typename TR::elem* __restrict__ out,
    float* __restrict__ lse, int H, int Sq, int Sk, float scale,
    GateArgs<typename TR::elem> ga, BiasMfma bm, FwdItems items) {
    static_assert(!BM || VEC, "the bias MFMA reads the bias tile from LDS");
    static_assert(!ODD || (VEC && !BM), "odd key counts run the plain form, the bias in LDS");
    static_assert(!(NSHD && GATE), "the gated entry takes the [N, H, S, D] layout");
    using E = typename TR::elem;
    using V8 = typename TR::vec8;
    using G = AttnGeom<D>;
    using T = SwzTile<D>;
    // PATCH (the bias tile in LDS): a key tile with an absent key (or keys past Sk) has its bias
    // changed in LDS before use -- a large negative bias for an absent key (P = 0 after the
    // exponential once the row's max comes from a present key): the masked logit -1e9 in
    // bfloat16, float16's lowest value -65504 in float16 (the reference's own masked logit is
    // -1e4) -- and the scores need no per-key select, so the tile's MFMAs and exponentials stay
    // one straight-line block. (A row without any present key computes no scores: tile_empty.)
    // (No larger magnitude: the exponent's FMA against the running max leaves a rounding residue of
    // about 2^-24 of the logit, which must stay far below float32's exponent range.) A float16 query
    // whose own logits lie that low is redone with -1e9 at absent keys, as below.
    constexpr bool PATCH = VEC;
    using PF = TilePrefetch<TR, QT>;
    constexpr int BQ = 4 * 16 * QT;
    constexpr int BK = G::BK;
    constexpr int TILE = BK * T::ROWB;  // bytes of one K or V tile
    constexpr int BTILE = VEC ? BQ * 128 : 0;  // bias tile: BQ query rows of 64 keys
    constexpr int QS = ODD ? 2 : 1;            // query step between a block's rows

    // Two K/V buffers as separate LDS objects: the compiler then knows that reads of one do not
    // wait for the direct-to-LDS loads into the other.
    __shared__ __attribute__((aligned(16))) char kv0[2 * TILE + BTILE];  // K rows, V rows, bias
    __shared__ __attribute__((aligned(16))) char kv1[2 * TILE + BTILE];

    // The arguments of the set-up in one round of scalar loads: left to itself the compiler loads
    // each where it is first needed, four rounds in a row before the first tile's loads go out.
    asm volatile("" ::"s"(q), "s"(k), "s"(v), "s"(bias), "s"(kmask), "s"(H), "s"(Sq), "s"(Sk),
                 "s"(items.outer.d), "s"(items.outer.m), "s"(items.outer.s), "s"(items.inner.d),
                 "s"(items.inner.m), "s"(items.inner.s), "s"(items.grp), "s"(gridDim.x));

    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int r16 = lane & 15, g = lane >> 4;
    // 1-D grid of (query tile, head, row) work items, placed so that each XCD runs a contiguous
    // range of them. grp == 0: query tile fastest, then the head, then the row -- the blocks of
    // one (row, query tile) read the same gate rows of x and, in the [N, S, H, D] layout, the
    // same cache lines of q, k and v, and the query tiles of one (row, head) the same K and V.
    // grp > 0 (a bias too large to stay in an XCD's L2 over all heads): the head outermost, then
    // groups of grp rows, then the query tile, then the row within its group -- an XCD's resident
    // blocks then read one head's bias rows (the same for every row n) and the K and V of a few
    // rows, both of which stay in its L2.
    // ODD: the even and the odd queries of a range of 2*BQ are neighbouring work items.
    const int item = xcd_contiguous(blockIdx.x, gridDim.x);
    const int a = div_by(item, items.outer), rem = item - a * items.outer.d;
    const int b = div_by(rem, items.inner), at = rem - b * items.inner.d;
    int q0 = at, h = b, n = a;  // grp == 0
    if (items.grp > 0) {
        const int nb = b * items.grp;
        const FastDiv rows = items.nrows - nb < items.grp ? items.last_rows : items.rows;
        h = a;
        q0 = div_by(at, rows);
        n = nb + at - q0 * rows.d;
    }
    q0 = ODD ? (q0 >> 1) * 2 * BQ + (q0 & 1) : q0 * BQ;
    const size_t nh = (uint32_t)(n * H + h);  // below 2^31 (validate_attention)
    // Rows of one (n, h) in q, k, v and out: [N, H, S, D] (rows D apart), or with NSHD
    // [N, S, H, D] (rows H*D apart, head h at column block h).
    const int ld = NSHD ? H * D : D;
    const E* qp = q + (NSHD ? ((size_t)n * Sq * H + h) * D : nh * (uint32_t)Sq * D);
    const E* kp = k + (NSHD ? ((size_t)n * Sk * H + h) * D : nh * (uint32_t)Sk * D);
    const E* vp = v + (NSHD ? ((size_t)n * Sk * H + h) * D : nh * (uint32_t)Sk * D);
    E* const op = out ? out + (NSHD ? ((size_t)n * Sq * H + h) * D : nh * (uint32_t)Sq * D) : nullptr;
    const E* bp = bias + (size_t)(uint32_t)h * (uint32_t)Sq * (uint32_t)Sk;
    const uint8_t* mp = kmask ? kmask + (size_t)(uint32_t)n * (uint32_t)Sk : nullptr;
    const int qbase = q0 + wave * 16 * QT * QS;
    // Keys the block's tiles start before key 0 (0 or 1; every row of the block agrees).
    const int shift = ODD ? (h * Sq + q0) & 1 : 0;
    const int ntiles = (Sk + shift + BK - 1) / BK;

    // The Sk rows of (n, h): rows past Sk read zeros.
    const uint32_t kvbytes = NSHD ? (Sk > 0 ? (uint32_t)(((size_t)(Sk - 1) * ld + D) * 2) : 0u)
                                  : (uint32_t)Sk * D * 2;
    const Rsrc rk = buffer_rsrc(kp, kvbytes);
    const Rsrc rv = buffer_rsrc(vp, kvbytes);
    // The block's bias rows (queries q0 + QS*i, i < BQ, that exist), from `shift` keys before the
    // first. Its end is rounded up to a dword (loads are range-checked by dword): for ODD the bias
    // of all heads is an even number of elements, so that dword lies inside it.
    const int brows = min(BQ, (Sq - q0 + QS - 1) / QS);
    const Rsrc rb = buffer_rsrc(bp + (size_t)(uint32_t)q0 * (uint32_t)Sk - shift,
                                brows > 0 ? (uint32_t)((((brows - 1) * QS * Sk + Sk + shift) * 2 + 3) & ~3)
                                          : 0u);
    // Head h's D columns of the gate weight: row c (channel) starts HD elements after row c-1.
    const Rsrc rw = GATE ? buffer_rsrc(ga.wg + h * D, (uint32_t)((ga.C - 1) * ga.HD + D) * 2)
                         : rb;
    auto stage = [&](int k0, char* kv) {
        if (ODD && k0 == 0) {  // row -1 (shift = 1) reads zeros
            stage_rows_from<D, BK, 256, true>(rk, -shift, ld, kv, threadIdx.x);
            stage_rows_from<D, BK, 256, true>(rv, -shift, ld, kv + TILE, threadIdx.x);
        } else if constexpr (NSHD) {
            stage_rows_ld<D, BK, 256, true>(rk, k0 - shift, ld, kv, threadIdx.x);
            stage_rows_ld<D, BK, 256, true>(rv, k0 - shift, ld, kv + TILE, threadIdx.x);
        } else {
            stage_rows<D, BK, 256, true>(rk, k0 - shift, kv);
            stage_rows<D, BK, 256, true>(rv, k0 - shift, kv + TILE);
        }
        if constexpr (VEC) {
            // The block's bias rows, keys k0 - shift .. + 63 as eight 16-byte pieces per row; piece
            // p of row r sits at position p ^ (r & 7), so a 16-row operand read is conflict-free.
            // Rows past Sq read zeros; keys past Sk (last tile) and key -1 read what lies there,
            // and are patched.
            const int row = threadIdx.x >> 3, piece = (threadIdx.x & 7) ^ (row & 7);
            const int voff = (row * QS * Sk + 8 * piece) * 2;
            // The later loads' offsets as sums with an opaque zero: held in registers through the
            // loop they cost the kernel two spilled ones.
            int step = 64 * QS * Sk;
            asm volatile("" : "+s"(step));
            char* const dst = kv + 2 * TILE + __builtin_amdgcn_readfirstlane(wave) * 1024;
#pragma unroll
            for (int i = 0; i < BQ * 8 / 256; ++i)
                buf_dma16(rb, voff + i * step, k0 * 2, dst + i * 4096);
        }
    };
    // PATCH: this wave's mask bytes of its first kPre key tiles (t = wave + 4*i; lane l: key
    // 64t + l - shift), loaded before anything else so that the presence words below wait for
    // them alone. Out of range (key -1 too, a negative offset) reads zero. (That lane's later keys
    // are the same register plus an instruction offset; the sum wraps at 32 bits, as tested.)
    constexpr int kPre = 4;
    uint32_t mb[kPre];
    if constexpr (PATCH) {
        const Rsrc rm = buffer_rsrc(mp ? (const void*)mp : (const void*)bp, mp ? (uint32_t)Sk : 0u);
#pragma unroll
        for (int i = 0; i < kPre; ++i) mb[i] = buf_ld1(rm, (wave + 4 * i) * BK + lane - shift);
    }
    // B operand Q^T: lane (query r16, group g) holds head dims 32*ks + 8*g + 0..7.
    V8 qf[QT][G::KS];
    const Rsrc rq = buffer_rsrc(qp, NSHD ? (uint32_t)(((size_t)(Sq - 1) * ld + D) * 2)
                                         : (uint32_t)Sq * D * 2);
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
        const int row = qbase + (qt * 16 + r16) * QS;
#pragma unroll
        for (int ks = 0; ks < G::KS; ++ks) {
            const int d0 = ks * 32 + g * 8;
            qf[qt][ks] = bits_as<V8>(buf_ld16(rq, d0 < D ? (row * ld + d0) * 2 : kNoRow));
        }
    }
    // (With no keys at all the resources are empty and the tile reads zeros.)
    stage(0, kv0);

    // Not PATCH: bias rows of the lane's queries (clamped inside [0, Sq)), keys 32c + 8g + 0..7
    // per tile.
    const E* brow[QT];
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) brow[qt] = bp + (size_t)min(qbase + qt * 16 + r16, Sq - 1) * Sk;
    PF ca, cb;
    if (!PATCH && ntiles > 0) ca.load(brow, mp, 0, g, Sk);
    // The mask row's tile flags, with the Q and first-tile loads already in flight (PATCH
    // reads the same facts from the presence words instead).
    const RowFlags rf = PATCH ? RowFlags{0ull, kMaskedLogit} : row_flags(mp, Sk);
    // PATCH: the row's presence bits, one 64-bit word per key tile (bit j: key 64t + j - shift
    // exists and is present; the launch keeps ntiles <= kPresWords), and per wave 1 + the last
    // of its tiles that holds a present key (0 if none).
    __shared__ unsigned long long pres[PATCH ? kPresWords : 1];
    __shared__ int wave_last[PATCH ? 4 : 1];
    if constexpr (PATCH) {
        int last = 0;
#pragma unroll
        for (int i = 0; i < kPre; ++i) {
            const int t = wave + 4 * i, kk = t * BK + lane - shift;
            const unsigned long long b = __ballot(mp ? mb[i] != 0u : kk >= 0 && kk < Sk);
            if (b != 0ull) last = t + 1;
            if (lane == 0) pres[t] = b;  // (past the last tile: no key, a zero nobody reads)
        }
        for (int t = wave + 4 * kPre; t < ntiles; t += 4) {
            const int kk = t * BK + lane - shift;
            const unsigned long long b = __ballot(kk < Sk && (mp == nullptr || mp[kk] != 0));
            if (b != 0ull) last = t + 1;
            if (lane == 0) pres[t] = b;
        }
        if (lane == 0) wave_last[wave] = last;
    }
    // PATCH: a row without any present key runs tile_empty below. Otherwise the key tiles after
    // the row's last present key (a padding tail) add P = 0 to O and l and are not run at all:
    // after the row's max is set their P underflows to 0.
    bool row_empty = false;
    int nrun = ntiles;  // key tiles the loop runs
    if constexpr (PATCH) {
        lds_barrier();  // the presence words and counts are visible (the loads stay in flight)
        const int last = max(max(wave_last[0], wave_last[1]), max(wave_last[2], wave_last[3]));
        row_empty = mp && last == 0;
        if (!row_empty) nrun = last;
    }
    // PATCH: lane (row r16 of each sub-tile, group g) changes 16-byte pieces 4c + g (keys
    // k0 + 32c + 8g + 0..7) of its rows of tile kt's bias: all its pieces are read, changed and
    // written back in one round.
    auto patch = [&](const char* kvc, int kt) {
        char* const bt = const_cast<char*>(kvc) + 2 * TILE;
        const float fill_bias = std::is_same<TR, BF16>::value ? kMaskedLogit : -65504.f;
        const uint32_t neg = (uint32_t)__builtin_bit_cast(uint16_t, TR::from_f(fill_bias)) * 0x10001u;
        u32x4* at[2][QT];
        u32x4 v[2][QT];
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int qt = 0; qt < QT; ++qt) {
                const int row = wave * 16 * QT + 16 * qt + r16;
                at[c][qt] = reinterpret_cast<u32x4*>(bt + row * 128 + 16 * ((4 * c + g) ^ (row & 7)));
                v[c][qt] = *at[c][qt];
            }
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            // (A row without any present key runs tile_empty, which reads no bias.)
            const uint32_t bits = reinterpret_cast<const uint32_t*>(pres)[2 * kt + c] >> (8 * g);
            // Dword i holds keys 2i, 2i+1 (low, high half): keep the bias of present keys.
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint32_t keep = ((bits >> (2 * i)) & 1u ? 0xffffu : 0u) |
                                      ((bits >> (2 * i + 1)) & 1u ? 0xffff0000u : 0u);
#pragma unroll
                for (int qt = 0; qt < QT; ++qt)
                    v[c][qt][i] = (v[c][qt][i] & keep) | (neg & ~keep);
            }
        }
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int qt = 0; qt < QT; ++qt) *at[c][qt] = v[c][qt];
        // The K rows of absent keys become zeros: whatever they hold, their logit is then the
        // changed bias alone. (Rows that do not exist are zeros already. Every wave does all rows:
        // its own reads then need no barrier, and nobody writes anything else.) As asm, because the
        // compiler would have a store it can see wait for the next tile's direct-to-LDS loads
        // (with the bias MFMA, 757 residues 568 -> 577 us and 598).
        const unsigned long long w = pres[kt];
        const int rem = Sk + shift - kt * BK;
        unsigned long long exist = rem >= 64 ? ~0ull : (1ull << rem) - 1ull;
        if (ODD && kt == 0 && shift) exist &= ~1ull;
        if (__builtin_amdgcn_readfirstlane(w != exist)) {
            const u32x4 zero = {0u, 0u, 0u, 0u};
            const uint32_t at0 = lds_addr(kvc) + lane * 16;
#pragma unroll
            for (int i = 0; i < T::PL; ++i)
                if (!((w >> ((64 * i + lane) / T::PL)) & 1ull))
                    asm volatile("ds_write_b128 %0, %1" ::"v"(at0 + i * 1024), "v"(zero) : "memory");
        }
    };
    // In the bias-MFMA form every score is in units of 1/scale of the logit (xs = scale*log2e
    // per unit); otherwise in logit units (xs = log2e).
    const float masked_logit = BM ? rf.masked_logit * bm.bscale : rf.masked_logit;
    const float xs = BM ? bm.cexp : kLog2e;
    // A operand [hi*I | lo*I] of the bias MFMA: lane (row r16, group g) holds columns
    // 8g .. 8g+7, so its one nonzero is element r16 % 8 when g % 2 == r16 / 8.
    V8 idn;
    if constexpr (BM) {
        const uint32_t v = (uint32_t)__builtin_bit_cast(uint16_t, TR::from_f(g < 2 ? bm.hi : bm.lo))
                           << (16 * (r16 & 1));
        const int at = (g & 1) == (r16 >> 3) ? (r16 & 7) >> 1 : -1;
        u32x4 bits;
#pragma unroll
        for (int i = 0; i < 4; ++i) bits[i] = i == at ? v : 0u;
        idn = bits_as<V8>(bits);
    }

    // Running max, and O^T plus one extra accumulator per sub-tile: the MFMA of an all-ones
    // A operand with P^T, i.e. the row sum of the (rounded) P that the P.V product uses.
    V8 ones;
#pragma unroll
    for (int j = 0; j < 8; ++j) ones[j] = TR::from_f(1.f);
    // The running max starts at half the masked logit: a tile whose keys are all absent (its
    // max the masked logit) then adds P = 0 exactly. Starting lower, the first such tile would
    // set the max, and P = exp2(x*xs - m*xs) of its keys would be the exponential of the FMA's
    // rounding residue (up to 2^6 at a logit of 1e9), which float16 cannot hold. In a row with
    // no present key every logit is the masked logit 0, the start.
    // Kept as nm = -m*xs, the exponent's offset itself: a tile's move test is one FMA, its
    // exponent FMAs take nm as it is, and lse = m*scale + ln(l) becomes -nm*ln2 + ln(l).
    float nm[QT];
    f32x4 acc[QT][G::DT], lsum[QT];
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
        nm[qt] = -(0.5f * masked_logit) * xs;
        lsum[qt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int dt = 0; dt < G::DT; ++dt) acc[qt][dt] = f32x4{0.f, 0.f, 0.f, 0.f};
    }

    // Float16's changed bias is no lower than a caller's may be (LOWEST): whether some tile had one.
    constexpr bool LOWEST = PATCH && !std::is_same<TR, BF16>::value;
    bool patched = false;
    // PLAIN (PATCH): the same tile with the bias as it is added to each score, and a select per
    // absent key, for blocks whose bias holds -inf (below).
    auto tile = [&](int kt, const char* kvc, char* kvn, PF& cur, PF& nxt, auto plain_tag) {
        constexpr bool PLAIN = decltype(plain_tag)::value;
        constexpr bool BMT = BM && !PLAIN;  // the bias through the MFMA
        const float xt = PLAIN ? kLog2e : xs;
        const int k0 = kt * BK;
        async_wait();
        __syncthreads();  // tile kt visible; every wave is done with the other buffer
        bool need_mask;
        if constexpr (PATCH) {
            const int rem = Sk + shift - k0;  // keys of the tile below Sk
            const unsigned long long full = rem >= 64 ? ~0ull : (1ull << rem) - 1ull;
            need_mask = (rem < 64) || pres[kt] != full;
        } else {
            need_mask = kt >= 64 || ((rf.bits >> kt) & 1ull) != 0ull;
        }
        if (kt + 1 < nrun) {
            stage(k0 + BK, kvn);
            if constexpr (!PATCH) nxt.load(brow, mp, k0 + BK, g, Sk);
        } else if constexpr (GATE) {
            // The last key tile leaves the other buffer free: the wg rows of the first
            // kGateChannels gate channels go there now, ready for the epilogue.
            int t = threadIdx.x;
            asm volatile("" : "+v"(t));
            stage_rows_ld<D, kGateChannels, 256>(rw, 0, ga.HD, kvn, t);
        }
        if (LOWEST) patched = patched || need_mask;
        // Each wave reads only its own rows of the bias tile: no barrier after the change.
        if (PATCH && !PLAIN && need_mask) {
            patch(kvc, kt);
            // Nothing of the tile's work is interleaved with the change (registers).
            __atomic_signal_fence(__ATOMIC_SEQ_CST);
        }
        V8 kf[4][G::KS];
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int ks = 0; ks < G::KS; ++ks)
                kf[t][ks] = swz_row_operand<V8, D>(kvc, BM ? 16 * t + r16 : perm_key(t, r16), ks, g);
        V8 vf[G::DT][2];
#pragma unroll
        for (int dt = 0; dt < G::DT; ++dt)
#pragma unroll
            for (int c = 0; c < 2; ++c)
                vf[dt][c] = BM ? swz_tr_operand_split<V8, D>(kvc + TILE, 32 * c, dt, r16, g)
                               : swz_tr_operand<V8, D>(kvc + TILE, 32 * c, dt, r16, g);

        // S^T = K . Q^T for the four 16-key sub-tiles (chunk c = t/2, half t%2).
        f32x4 s[QT][4];
        if constexpr (BMT) {
            // Bias / scale first. S^T tile t holds keys 16t + 0..15 of the key tile here, so
            // rows 8g' + j of the B operand (g' = g % 2, duplicated for the lo half) are keys
            // 16t + 8g' + 0..7 of the lane's query row: one 16-byte piece, 2t + g', of the
            // swizzled bias rows (piece p of row r at p ^ (r & 7)).
#pragma unroll
            for (int qt = 0; qt < QT; ++qt) {
                const int row = wave * 16 * QT + 16 * qt + r16;
                const char* brow_l = kvc + 2 * TILE + row * 128;
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    const u32x4 raw = *reinterpret_cast<const u32x4*>(
                        brow_l + 16 * ((2 * t + (g & 1)) ^ (row & 7)));
                    s[qt][t] = TR::mfma(idn, bits_as<V8>(raw), f32x4{0.f, 0.f, 0.f, 0.f});
                }
            }
        }
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int ks = 0; ks < G::KS; ++ks)
#pragma unroll
                for (int qt = 0; qt < QT; ++qt)
                    s[qt][t] = TR::mfma(kf[t][ks], qf[qt][ks],
                                        (BMT || ks > 0) ? s[qt][t] : f32x4{0.f, 0.f, 0.f, 0.f});

        float x[QT][2][8];
#pragma unroll
        for (int qt = 0; qt < QT; ++qt)
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                if constexpr (BM) {
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        x[qt][c][j] = s[qt][2 * c][j];
                        x[qt][c][4 + j] = s[qt][2 * c + 1][j];
                    }
                    if constexpr (PLAIN) {
                        // Keys 16t + 4g + 0..3 of the lane's query, t = 2c + u: half a piece.
                        const int row = wave * 16 * QT + 16 * qt + r16;
#pragma unroll
                        for (int u = 0; u < 2; ++u) {
                            E e[4];
                            __builtin_memcpy(e, kvc + 2 * TILE + row * 128 + 8 * (g & 1) +
                                                    16 * ((4 * c + 2 * u + (g >> 1)) ^ (row & 7)),
                                             8);
#pragma unroll
                            for (int j = 0; j < 4; ++j)
                                x[qt][c][4 * u + j] =
                                    fmaf(x[qt][c][4 * u + j], scale, TR::to_f(e[j]));
                        }
                    }
                    continue;
                }
                float bv[8];
                if constexpr (VEC) {
                    const int row = wave * 16 * QT + 16 * qt + r16;
                    unpack8<TR>(*reinterpret_cast<const u32x4*>(
                                    kvc + 2 * TILE + row * 128 + 16 * ((4 * c + g) ^ (row & 7))),
                                bv);
                } else {
                    unpack8<TR>(cur.bias[qt][c], bv);
                }
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    x[qt][c][j] = fmaf(s[qt][2 * c][j], scale, bv[j]);
                    x[qt][c][4 + j] = fmaf(s[qt][2 * c + 1][j], scale, bv[4 + j]);
                }
            }
        if (!PATCH && need_mask) {
            // One block for the whole tile, opaque to speculation: nothing of it is hoisted
            // into (or merged across sub-tiles onto) the unmasked path.
            asm volatile("");
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                // Slot j is key k0 + 32c + 8g + j.
                const int lim = Sk - (k0 + 32 * c + 8 * g);
                const unsigned valid = cur.valid(c);
#pragma unroll
                for (int qt = 0; qt < QT; ++qt)
#pragma unroll
                    for (int j = 0; j < 8; ++j)
                        x[qt][c][j] = j >= lim
                                          ? -INFINITY
                                          : (((valid >> j) & 1u) ? x[qt][c][j] : masked_logit);
            }
        }

        if constexpr (PLAIN) {
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                const uint32_t w = reinterpret_cast<const uint32_t*>(pres)[2 * kt + c];
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const int bit = !BM ? 8 * g + j : 4 * g + (j < 4 ? j : 12 + j);
#pragma unroll
                    for (int qt = 0; qt < QT; ++qt)
                        x[qt][c][j] = (w >> bit) & 1u ? x[qt][c][j] : kMaskedLogit;
                }
            }
        }

        float mt[QT];
#pragma unroll
        for (int qt = 0; qt < QT; ++qt) {
            mt[qt] = x[qt][0][0];
#pragma unroll
            for (int c = 0; c < 2; ++c)
#pragma unroll
                for (int j = 0; j < 8; ++j) mt[qt] = fmaxf(mt[qt], x[qt][c][j]);
        }
        if constexpr (QT == 2) {
            xgroup_max2(mt[0], mt[1]);
        } else {
#pragma unroll
            for (int qt = 0; qt < QT; ++qt) mt[qt] = xgroup_max(mt[qt]);
        }
#pragma unroll
        for (int qt = 0; qt < QT; ++qt) {
            // Lazy rescaling: the running max moves only when the tile's max exceeds it by more
            // than kRescaleSlack (in log2 units), so P stays below 2^kRescaleSlack and most tiles
            // skip the rescale of O and l (a wave-uniform branch).
            const bool move = fmaf(mt[qt], xt, nm[qt]) > kRescaleSlack;
            if (__any(move)) {
                // Opaque to if-conversion: without it the compiler runs the rescale on every
                // tile (alpha = 1 when nothing moved gives the same values).
                asm volatile("");
                const float nm_new = move ? -mt[qt] * xt : nm[qt];
                const float alpha = fast_exp2(nm_new - nm[qt]);
                nm[qt] = nm_new;
                lsum[qt][0] *= alpha;  // only component 0 is read
#pragma unroll
                for (int dt = 0; dt < G::DT; ++dt) acc[qt][dt] *= alpha;
            }
            const float neg = nm[qt];
            V8 pf[2];
#pragma unroll
            for (int c = 0; c < 2; ++c)
#pragma unroll
                for (int j = 0; j < 8; ++j) pf[c][j] = TR::from_f(fast_exp2(fmaf(x[qt][c][j], xt, neg)));
#pragma unroll
            for (int c = 0; c < 2; ++c) lsum[qt] = TR::mfma(ones, pf[c], lsum[qt]);
#pragma unroll
            for (int dt = 0; dt < G::DT; ++dt)
#pragma unroll
                for (int c = 0; c < 2; ++c) acc[qt][dt] = TR::mfma(vf[dt][c], pf[c], acc[qt][dt]);
        }
    };
    // PATCH, a row without any present key: every logit in range is the masked logit 0, so
    // P = 1 there (and 0 past Sk) with the running max at 0 -- the values the tiles above
    // compute for such a row -- and a tile needs only its V rows: no S, no exponential.
    auto tile_empty = [&](int kt, const char* kvc, char* kvn) {
        const int k0 = kt * BK;
        async_wait();
        __syncthreads();  // tile kt visible; every wave is done with the other buffer
        if (kt + 1 < nrun) {
            stage(k0 + BK, kvn);
        } else if constexpr (GATE) {
            int t = threadIdx.x;
            asm volatile("" : "+v"(t));
            stage_rows_ld<D, kGateChannels, 256>(rw, 0, ga.HD, kvn, t);
        }
        V8 vf[G::DT][2];
#pragma unroll
        for (int dt = 0; dt < G::DT; ++dt)
#pragma unroll
            for (int c = 0; c < 2; ++c)
                vf[dt][c] = BM ? swz_tr_operand_split<V8, D>(kvc + TILE, 32 * c, dt, r16, g)
                               : swz_tr_operand<V8, D>(kvc + TILE, 32 * c, dt, r16, g);
        // Slot j of chunk c is key k0 - shift + 32c + 8g + j, or in the bias-MFMA order
        // k0 - shift + 32c + 4g + j (j < 4) and k0 - shift + 32c + 12 + 4g + j (j >= 4). (Key -1,
        // the first slot of lane group 0 in tile 0 when shift = 1, has P = 0.)
        V8 pf[2];
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            const int lim = Sk + shift - (k0 + 32 * c + (BM ? 4 : 8) * g);
#pragma unroll
            for (int j = 0; j < 8; ++j)
                pf[c][j] = TR::from_f((BM && j >= 4 ? j + 12 : j) < lim ? 1.f : 0.f);
        }
        if (ODD && k0 == 0 && g == 0 && shift) pf[0][0] = TR::from_f(0.f);
#pragma unroll
        for (int qt = 0; qt < QT; ++qt) {
#pragma unroll
            for (int c = 0; c < 2; ++c) lsum[qt] = TR::mfma(ones, pf[c], lsum[qt]);
#pragma unroll
            for (int dt = 0; dt < G::DT; ++dt)
#pragma unroll
                for (int c = 0; c < 2; ++c) acc[qt][dt] = TR::mfma(vf[dt][c], pf[c], acc[qt][dt]);
        }
    };
    if (PATCH && row_empty) {  // block-uniform
#pragma unroll
        for (int qt = 0; qt < QT; ++qt) nm[qt] = 0.f;
        for (int kt = 0; kt < nrun; kt += 2) {
            tile_empty(kt, kv0, kv1);
            if (kt + 1 < nrun) tile_empty(kt + 1, kv1, kv0);
        }
    } else {
        for (int kt = 0; kt < nrun; kt += 2) {
            tile(kt, kv0, kv1, ca, cb, std::false_type{});
            if (kt + 1 < nrun) tile(kt + 1, kv1, kv0, cb, ca, std::false_type{});
        }
        if constexpr (BM || LOWEST) {
            // A bias of -inf leaves NaN in the row sum of its query (the zeros of the bias MFMA's
            // operand times it are NaN). A block with one redoes its keys in the plain form, where
            // -inf is a weight of 0. So does a float16 block with a row maximum near -65504, where
            // absent keys would take weight: above -65400 theirs is below float32's smallest number.
            // (NaN by its bits: this file is compiled without NaN semantics. The look at the sums
            // and its barrier: 384 residues 269.8 -> 271.0 us, 1024 with the gate 1167 -> 1173,
            // 1024 x 300 at D = 8 262.9 -> 266.0.)
            bool bad = false;
#pragma unroll
            for (int qt = 0; qt < QT; ++qt) {
                bad = bad || (__float_as_uint(lsum[qt][0]) & 0x7fffffffu) > 0x7f800000u;
                if (LOWEST) bad = bad || (patched && nm[qt] > 65400.f * kLog2e);
            }
            const bool wave_bad = __any(bad);
            if (lane == 0) wave_last[wave] = wave_bad;
            lds_barrier();
            const int any_bad = (wave_last[0] | wave_last[1]) | (wave_last[2] | wave_last[3]);
            if (__builtin_amdgcn_readfirstlane(any_bad)) {
                async_wait();
                __syncthreads();  // no load into a buffer is in flight, no wave reads one
#pragma unroll
                for (int qt = 0; qt < QT; ++qt) {
                    nm[qt] = -(0.5f * kMaskedLogit) * kLog2e;
                    lsum[qt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int dt = 0; dt < G::DT; ++dt) acc[qt][dt] = f32x4{0.f, 0.f, 0.f, 0.f};
                }
                stage(0, kv0);
#pragma unroll 1
                for (int kt = 0; kt < nrun; ++kt)
                    tile(kt, kt & 1 ? kv1 : kv0, kt & 1 ? kv0 : kv1, ca, cb, std::true_type{});
            }
        }
    }
    if (nrun == 0) async_wait();  // no keys: tile 0's loads end before the block (or its gate)

    // Gate pre-activations in O^T's accumulator layout (lane: rows 16*dt + 4*g + i of head h's
    // columns, query r16), so gate and O pair up element for element.
    f32x4 gacc[GATE ? QT : 1][G::DT];
    if constexpr (GATE) {
        // G^T = Wg_h^T . X^T + bg_h, 2*kGateChannels channels per round: A = head h's wg
        // columns for kGateChannels channels per K/V buffer (both buffers hold 128 rows of D),
        // staged like a V tile and read transposed; B = eight consecutive channels of the
        // lane's query row of x, straight from global memory into registers (zero for rows past
        // Sq and channels past C). The first buffer's rows were fetched during the last key
        // tile, and the x loads are issued before the barrier, so a round costs one wait.
        const int C = ga.C, HD = ga.HD;
        // Thread coordinates recomputed from an opaque copy of the thread index: shared with
        // the key loop, the epilogue's offsets would stay live (in registers) through it.
        int tid = threadIdx.x;
        asm volatile("" : "+v"(tid));
        const int gr16 = tid & 15, gg = (tid >> 4) & 3;
#pragma unroll
        for (int dt = 0; dt < G::DT; ++dt) {
            const int d = 16 * dt + 4 * gg;
            f32x4 b0 = {0.f, 0.f, 0.f, 0.f};
            if (d < D)
#pragma unroll
                for (int i = 0; i < 4; ++i) b0[i] = TR::to_f(ga.bg[h * D + d + i]);
#pragma unroll
            for (int qt = 0; qt < QT; ++qt) gacc[qt][dt] = b0;
        }
        constexpr int GC = kGateChannels, NX = 2 * GC / 32;
        static_assert(GC * T::ROWB <= 2 * TILE, "a K/V buffer holds kGateChannels wg rows");
        char* const kfree = (nrun & 1) ? kv1 : kv0;  // not read by the last key tile
        char* const klast = (nrun & 1) ? kv0 : kv1;
        for (int c0 = 0; c0 < C; c0 += 2 * GC) {
            V8 xo[QT][NX];
#pragma unroll
            for (int qt = 0; qt < QT; ++qt) {
                const int row = q0 + (16 * QT * (tid >> 6) + qt * 16 + gr16) * QS;
#pragma unroll
                for (int j = 0; j < NX; ++j) {
                    const int c = c0 + 32 * j;
                    u32x4 raw = {0u, 0u, 0u, 0u};
                    if (c < C && row < Sq)
                        raw = ld16(ga.x + ((size_t)n * Sq + row) * C + c + 8 * gg);
                    xo[qt][j] = bits_as<V8>(raw);
                }
            }
            __syncthreads();  // every wave is done with both buffers
            if (c0 > 0 || nrun == 0) stage_rows_ld<D, GC, 256>(rw, c0, HD, kfree, tid);
            if (c0 + GC < C) stage_rows_ld<D, GC, 256>(rw, c0 + GC, HD, klast, tid);
            async_wait();
            __syncthreads();  // this round's wg rows are visible
#pragma unroll
            for (int half = 0; half < 2; ++half)
#pragma unroll
                for (int cc = 0; cc < GC / 32; ++cc) {
                    if (c0 + GC * half + 32 * cc >= C) break;  // wave-uniform
#pragma unroll
                    for (int dt = 0; dt < G::DT; ++dt) {
                        const V8 a =
                            swz_tr_operand<V8, D>(half ? klast : kfree, 32 * cc, dt, gr16, gg);
#pragma unroll
                        for (int qt = 0; qt < QT; ++qt)
                            gacc[qt][dt] = TR::mfma(a, xo[qt][(GC / 32) * half + cc], gacc[qt][dt]);
                    }
                }
        }
    }

    // Normalise and store: lane holds O[row][16*dt + 4*g + i], i = 0..3. With the gate, O is
    // stored only when `out` is given, and the gated row goes to its [N, Sq, HD] place (its
    // lane coordinates again from an opaque thread index, as in the gate products).
    int etid = threadIdx.x;
    if constexpr (GATE) asm volatile("" : "+v"(etid));
    const int er16 = etid & 15, eg = (etid >> 4) & 3;
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
        const float l_tot = lsum[qt][0];
        const float inv = 1.0f / fmaxf(l_tot, 1e-30f);
        const int row = q0 + (16 * QT * (etid >> 6) + qt * 16 + er16) * QS;
        if (row >= Sq) continue;
#pragma unroll
        for (int dt = 0; dt < G::DT; ++dt) {
            const int d = 16 * dt + 4 * eg;
            if (d >= D) continue;
            const f32x4 o = acc[qt][dt] * inv;
            if (!GATE || out) store4<TR>(op + (size_t)row * ld + d, o);
            if constexpr (GATE) {
                f32x4 r;
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    r[i] = o[i] * fast_rcp(1.f + fast_exp2(-kLog2e * gacc[qt][dt][i]));
                store4<TR>(ga.gated + ((size_t)n * Sq + row) * ga.HD + h * D + d, r);
            }
        }
        // A row whose present-key logits all lie below the running max's start (half the masked
        // logit) has no weight: O = 0 and lse = +inf, so the backward's P is 0 there.
        if (lse && eg == 0)
            lse[nh * Sq + row] =
                l_tot > 0.f ? -nm[qt] * kLn2 + logf(l_tot) : INFINITY;
    }
}

// How a call's bias reaches the kernel.
struct FwdForm {
    BiasMfma bm{};
    bool bmf, odd, vec;
};

// Most blocks of a launch: a grid is at most 2^32 - 1 threads (more wrap around, without an error).
constexpr int64_t kMaxBlocks = (((int64_t)1 << 32) - 1) / 256;

// Query blocks of one (row, head) at 64*QT queries each.
int fwd_qtiles(bool odd, int Sq, int QT) {
    return odd ? 2 * ceil_div((Sq + 1) / 2, 64 * QT) : ceil_div(Sq, 64 * QT);
}

// The bias tile through LDS (vec: direct loads of 4-byte aligned pieces): at most kPresWords key
// tiles (masked bias tiles are changed in LDS from presence words kept there). An even Sk
// aligns every bias row. An odd one takes the parity form, when the bias is a whole number of
// dwords (no load then reaches past its end). Other odd cases (one head or an odd number of them
// with an odd Sq, so many short rows that two parities of blocks pass the largest launch) and longer
// rows read bias and mask element by element, about four times slower (2395
// against 529 us at 757 residues).
//
// Multiples of 8 take the bias MFMA (two VALU instructions a score less, 1-2% of the time). Ragged
// counts add the bias to each score as the element-wise path does, exact in float32; a bias MFMA
// that is (a third 16-bit term of 1/scale in bfloat16, cexp that of the pair in float16) is slower:
// 757 residues at D = 32 566 against 529 us in bfloat16, 542 against 530 in float16, 1024 x 300 at
// D = 8 281 against 257 and 263 against 255; D = 16, whose 1/scale is one value, 96 against 101.
template <typename TR>
FwdForm fwd_form(int64_t NH, int H, int Sq, int Sk, float scale) {
    FwdForm f;
    f.bmf = Sk % 8 == 0 && bias_mfma_for<TR>(scale, &f.bm);
    const bool odd = Sk % 2 && (size_t)H * Sq * Sk % 2 == 0 &&
                     NH * fwd_qtiles(true, Sq, Sq <= 64 ? 1 : 2) <= kMaxBlocks;
    f.vec = (Sk % 2 == 0 || odd) && Sk + (odd ? 1 : 0) <= kPresWords * 64;
    f.odd = f.vec && odd;
    return f;
}

// Queries per block: 64 (one 16-query sub-tile a wave) or 128 (two, which share each K, V and
// presence read). Per query the smaller block costs 0-3% more time at D <= 16, 10% at D = 32 and
// 40% at D = 64, so it is taken (us, smaller against larger block, bf16)
//  - where its finer rounding saves more than that: an odd number m of 64-query tiles (m + 1 are
//    run otherwise) at D <= 16, and m <= 7 at D = 32. D = 8, 300 queries 270 against 297; D = 16,
//    300 38.6 against 47.5, 400 83 against 99; D = 32, 192 15.8 / 17.1, 300 47.4 / 50.8, 400
//    110.4 / 111.9, but 704 116 / 114. An even m: 512 135 / 137 at D = 16, 182 / 163 at D = 32.
//  - where all the smaller blocks are resident at once, so that a call lasts one block and half
//    the block is nearly half the time: 4 per CU, 2 at D = 64 (gated, D = 32, 1024 blocks 11.9
//    against 15.0, but 1536 16.7 / 15.3; D = 64, 512 blocks 13.1 / 15.7, but 768 17.4 / 15.8).
bool fwd_small_blocks(const FwdForm& f, int D, int64_t NH, int Sq) {
    if (Sq <= 64) return true;
    if (!f.vec) return false;
    const int m = fwd_qtiles(f.odd, Sq, 1);
    if (NH * m > kMaxBlocks) return false;
    if (NH * m <= (D == 64 ? 512 : 1024)) return true;
    return m < 2 * fwd_qtiles(f.odd, Sq, 2) && (D <= 16 || (D == 32 && m <= 7));
}

template <typename TR, int D, int QT, bool GATE, bool NSHD>
void launch_fwd_qt(hipStream_t st, const void* q, const void* k, const void* v, const void* bias,
                   const uint8_t* kmask, void* out, float* lse, int N, int H, int Sq, int Sk,
                   float scale, GateArgs<typename TR::elem> ga, const FwdForm& f) {
    using E = typename TR::elem;
    const int qtiles = fwd_qtiles(f.odd, Sq, QT);
    const dim3 grid(qtiles * H * N);
    // The head-outer work-item order when the bias of all heads passes half of an XCD's 4 MB L2,
    // in groups of rows whose query tiles make about 48 work items, half an XCD's resident
    // blocks (32 CUs x 3): at N_res = 1024 (8 MB of bias) this cut the launch's fetch from 8.2 to
    // 0.9 GB and its time by 9% (any group of 4 to 24 rows within 1%). Otherwise the head stays
    // inside the row: the MSA shapes' gate rows and [N, S, H, D] rows are shared by the heads.
    const bool head_outer = (size_t)H * Sq * Sk * 2 > (2u << 20);
    const int grp = head_outer ? max(1, min(N, 48 / qtiles)) : 0;
    FwdItems items{};
    items.grp = grp;
    items.nrows = N;
    items.outer = fast_div(qtiles * (grp ? N : H));
    items.inner = fast_div(qtiles * (grp ? grp : 1));
    items.rows = fast_div(grp ? grp : 1);
    items.last_rows = fast_div(grp && N % grp ? N % grp : max(1, grp));
    auto run = [&](auto kernel) {
        kernel<<<grid, 256, 0, st>>>((const E*)q, (const E*)k, (const E*)v, (const E*)bias, kmask,
                                     (E*)out, lse, H, Sq, Sk, scale, ga, f.bm, items);
    };
    if (f.odd)
        run(attn_fwd_kernel<TR, D, QT, true, GATE, false, NSHD, true>);
    else if (f.vec && f.bmf)
        run(attn_fwd_kernel<TR, D, QT, true, GATE, true, NSHD, false>);
    else if (f.vec)
        run(attn_fwd_kernel<TR, D, QT, true, GATE, false, NSHD, false>);
    else
        run(attn_fwd_kernel<TR, D, QT, false, GATE, false, NSHD, false>);
}

template <typename TR, int D, bool GATE>
void launch_fwd(hipStream_t st, const void* q, const void* k, const void* v, const void* bias,
                const uint8_t* kmask, void* out, float* lse, int N, int H, int Sq, int Sk,
                float scale, GateArgs<typename TR::elem> ga, int nshd) {
    KernelTimer timer(GATE ? "attn_fwd_gated" : "attn_fwd", st);
    const FwdForm f = fwd_form<TR>((int64_t)N * H, H, Sq, Sk, scale);
    const bool small = fwd_small_blocks(f, D, (int64_t)N * H, Sq);
    auto launch = [&](auto qt, auto rows_nshd) {
        launch_fwd_qt<TR, D, decltype(qt)::value, GATE, decltype(rows_nshd)::value>(
            st, q, k, v, bias, kmask, out, lse, N, H, Sq, Sk, scale, ga, f);
    };
    using One = std::integral_constant<int, 1>;
    using Two = std::integral_constant<int, 2>;
    // The [N, S, H, D] layout only for the ungated forward.
    if constexpr (!GATE) {
        if (nshd) {
            if (small) launch(One{}, std::true_type{});
            else launch(Two{}, std::true_type{});
            return;
        }
    }
    if (small) launch(One{}, std::false_type{});
    else launch(Two{}, std::false_type{});
}

template <typename TR, bool GATE>
void dispatch_fwd(hipStream_t st, int64_t D, const void* q, const void* k, const void* v,
                  const void* bias, const uint8_t* kmask, void* out, float* lse, int N, int H,
                  int Sq, int Sk, float scale, GateArgs<typename TR::elem> ga, int nshd = 0) {
    switch (D) {
#define CLK_FWD_D(DV)                                                                           \
    case DV:                                                                                    \
        launch_fwd<TR, DV, GATE>(st, q, k, v, bias, kmask, out, lse, N, H, Sq, Sk, scale, ga,   \
                                 nshd);                                                         \
        break;
        CLK_FWD_D(8) CLK_FWD_D(16) CLK_FWD_D(32)
#undef CLK_FWD_D
        default:
            launch_fwd<TR, 64, GATE>(st, q, k, v, bias, kmask, out, lse, N, H, Sq, Sk, scale, ga,
                                     nshd);
            break;
    }
}

template <typename TR>
GateArgs<typename TR::elem> gate_args(const void* x, const void* wg, const void* bg, void* gated,
                                      int C, int HD) {
    using E = typename TR::elem;
    return {(const E*)x, (const E*)wg, (const E*)bg, (E*)gated, C, HD};
}

}  // namespace
}  // namespace clk

using namespace clk;

extern "C" clk_status clk_attention_fwd(hipStream_t stream, clk_dtype dtype, const void* q,
                                        const void* k, const void* v, const void* bias,
                                        const uint8_t* kmask, void* out, float* lse, int64_t N,
                                        int64_t H, int64_t Sq, int64_t Sk, int64_t D, float scale,
                                        int64_t block_q, int64_t block_k) {
    clk_status s = validate_attention("attention", dtype, N, H, Sq, Sk, D);
    if (s != CLK_OK) return s;
    if (block_q <= 0 || block_k <= 0)
        return fail(CLK_INVALID_ARGUMENT, "attention: block_q and block_k must be positive");
    if (N * H * Sq == 0) return ok();
    if (!q || !k || !v || !bias || !out)
        return fail(CLK_INVALID_ARGUMENT, "attention: null operand pointer");
    if (!aligned16(q) || !aligned16(k) || !aligned16(v) || !aligned16(bias) || !aligned16(out))
        return fail(CLK_INVALID_ARGUMENT, "attention: q, k, v, bias, out must be 16-byte aligned");
    if (dtype == CLK_BF16)
        dispatch_fwd<BF16, false>(stream, D, q, k, v, bias, kmask, out, lse, (int)N, (int)H,
                                  (int)Sq, (int)Sk, scale, {});
    else
        dispatch_fwd<F16, false>(stream, D, q, k, v, bias, kmask, out, lse, (int)N, (int)H,
                                 (int)Sq, (int)Sk, scale, {});
    return check_launch("attention");
}

extern "C" clk_status clk_attention_fwd_nshd(hipStream_t stream, clk_dtype dtype, const void* q,
                                             const void* k, const void* v, const void* bias,
                                             const uint8_t* kmask, void* out, float* lse,
                                             int64_t N, int64_t H, int64_t Sq, int64_t Sk,
                                             int64_t D, float scale) {
    const char* who = "attention_nshd";
    clk_status s = validate_attention(who, dtype, N, H, Sq, Sk, D);
    if (s != CLK_OK) return s;
    // Byte offsets within the rows of one (n, h) are 32-bit: S*H*D*2 below 2^31.
    if ((Sq > Sk ? Sq : Sk) * H * D * 2 >= ((int64_t)1 << 31))
        return fail(CLK_INVALID_ARGUMENT, "%s: S*H*D too large for the [N,S,H,D] layout", who);
    if (N * H * Sq == 0) return ok();
    if (!q || !k || !v || !bias || !out)
        return fail(CLK_INVALID_ARGUMENT, "%s: null operand pointer", who);
    if (!aligned16(q) || !aligned16(k) || !aligned16(v) || !aligned16(bias) || !aligned16(out))
        return fail(CLK_INVALID_ARGUMENT, "%s: q, k, v, bias, out must be 16-byte aligned", who);
    if (dtype == CLK_BF16)
        dispatch_fwd<BF16, false>(stream, D, q, k, v, bias, kmask, out, lse, (int)N, (int)H,
                                  (int)Sq, (int)Sk, scale, {}, 1);
    else
        dispatch_fwd<F16, false>(stream, D, q, k, v, bias, kmask, out, lse, (int)N, (int)H,
                                 (int)Sq, (int)Sk, scale, {}, 1);
    return check_launch(who);
}

extern "C" clk_status clk_attention_fwd_gated(hipStream_t stream, clk_dtype dtype, const void* q,
                                              const void* k, const void* v, const void* bias,
                                              const uint8_t* kmask, const void* x, const void* wg,
                                              const void* bg, void* gated, void* out, float* lse,
                                              int64_t N, int64_t H, int64_t Sq, int64_t Sk,
                                              int64_t D, int64_t C, float scale) {
    const char* who = "attention_gated";
    clk_status s = validate_attention(who, dtype, N, H, Sq, Sk, D);
    if (s != CLK_OK) return s;
    if (C <= 0 || C % 32)
        return fail(CLK_INVALID_ARGUMENT, "%s: C=%lld must be a positive multiple of 32", who,
                    (long long)C);
    const int64_t HD = H * D;
    // Buffer offsets into a row block of x and into wg are 32-bit.
    if (Sq * C * 2 >= ((int64_t)1 << 30) || C * HD * 2 >= ((int64_t)1 << 30))
        return fail(CLK_INVALID_ARGUMENT, "%s: Sq*C or C*H*D too large", who);
    if (N * H * Sq == 0) return ok();
    if (!q || !k || !v || !bias || !x || !wg || !bg || !gated)
        return fail(CLK_INVALID_ARGUMENT, "%s: null operand pointer", who);
    if (!aligned16(q) || !aligned16(k) || !aligned16(v) || !aligned16(bias) || !aligned16(x) ||
        !aligned16(wg) || !aligned16(gated) || (out && !aligned16(out)))
        return fail(CLK_INVALID_ARGUMENT,
                    "%s: q, k, v, bias, x, wg, gated, out must be 16-byte aligned", who);
    if (dtype == CLK_BF16)
        dispatch_fwd<BF16, true>(stream, D, q, k, v, bias, kmask, out, lse, (int)N, (int)H,
                                 (int)Sq, (int)Sk, scale,
                                 gate_args<BF16>(x, wg, bg, gated, (int)C, (int)HD));
    else
        dispatch_fwd<F16, true>(stream, D, q, k, v, bias, kmask, out, lse, (int)N, (int)H,
                                (int)Sq, (int)Sk, scale,
                                gate_args<F16>(x, wg, bg, gated, (int)C, (int)HD));
    return check_launch(who);
}
