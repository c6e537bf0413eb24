// Paged causal / chunked / non-causal prefill attention, ping-pong form (gfx950, bf16
// MFMA, dense bf16 or INT8 cache, head_dim 64 or 128, power-of-two pages of >= 16 tokens).
//
// Reference: attention_prefill_kernel / prefill_body (src/ops/tile/attention.jl:130-177)
// and attention_prefill_int8_kernel (:139-147). Query t of the step sits at position
// start + t (start = positions of the sequence's first query, read on the device) and sees
// keys 0 .. start + t; with causal = 0 it sees all start + n keys (attention.jl:155-157).
//
// A work-group is one or two teams of 4 waves (team A = waves 0-3, team B = waves 4-7; wave w
// runs on SIMD w % 4, so each SIMD holds one wave of each team). Every wave owns 32 packed
// query rows. With two teams, work-group barriers split time into phases; in every phase one team runs its
// MFMAs while the other runs its softmax, so each SIMD's matrix core and VALU work at the
// same time. Team B runs one phase behind team A:
//
//   phase      0      1      2      3      4     ...
//   team A    X0     Y0     X1     Y1     X2
//   team B    --     X0     Y0     X1     Y1
//
//   X_i = S_i = K_i Q^T and O += V_{i-1} P_{i-1}, and in the MFMAs' shadow everything else
//         that is not softmax: V operands of tile i - 1 and K operands of tile i + 1 from
//         LDS, staged tiles into LDS, global loads of later tiles
//   Y_i = online softmax of S_i -> P_i (bf16), lazy rescale of O
//
// Three forms (ti_pick_prefill_pp below has the rule and the figures):
//   SHARED  all 8 waves share each 32-key tile (256 packed rows per work-group);
//   KSPLIT  both teams hold the same 128 rows and take every other tile each (team t: tiles
//           t, t + 2, ...), merged through LDS at the end: half the rows per work-group and
//           half the steps, for launches whose 256-row tiles leave CUs idle;
//   SOLO    one team on 128 rows, one barrier a step; two work-groups (head_dim 64: three)
//           share a CU and overlap each other's phases, first loads and stores.
//
// What bounds it: the two phases and the clock. In steady replays at 8192 tokens the chip runs this
// kernel at 1.87 GHz (cycle counter over the real-time counter, per work-group; 4096 tokens 1.90;
// a loop of these MFMAs alone 1.5-1.7, one on 8 CUs 2.4), and a SHARED step takes 0.87 us, of
// which its MFMAs (8 waves x 16 of 32 cycles, 1024 cycles a SIMD) fill 63 %; softmax phases and
// barriers, not told apart, keep the matrix cores waiting for the rest. Work-groups are busy 455 of
// the call's 492 us. The MFMA phase used to wait for its operands: keys read in pairs just
// before their MFMAs, softmax phases carrying the staging. With the keys' operands read a phase
// ahead, the values' behind the first scores, score and value MFMAs taking turns and everything
// else in the gaps between them: 8192 tokens 539 -> 493 us (1115 TFLOP/s; bf16 GEMMs of this size
// reach 1350-1600 here), 4096 tokens 146 -> 135, 2000 on 4000 204 -> 165 (same process, graph
// replays, inputs of unit variance).
//
// The per-wave MFMA layouts, the exp2-domain online softmax with lazy rescale, the
// transposing V reads and the output / split-partial formats are those of the
// four-wave prefill kernel (pa_prefill.hip).
#include <stdlib.h>

#include <type_traits>

#include "common.hpp"

using namespace ti;

namespace {

constexpr int KT = 32;                 // keys per tile
constexpr float RESCALE_LOG2 = 8.0f;   // lazy-rescale threshold

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef short s16x4 __attribute__((ext_vector_type(4)));

struct PPParams {
    const uint16_t *q;
    uint16_t *out;
    const uint16_t *kp, *vp;
    const int8_t *lq;
    const float *ls, *smooth;
    const int32_t *positions, *qsl, *bt;
    float *part;                       // split partials [B][Hk][splits][M][D + 2]
    int bt_stride, num_pages, P, pshift, Hk, Hq, G, TQ, nmax, qtiles, causal, splits, sshift, M;   // splits = 2^sshift
    int eager;                         // first steps that rescale to every larger maximum
    float scale_log2;
};

// One tile stream's double-buffered tiles. Row strides (bf16): D + 8 for K (16-B reads by 16
// keys hit 64 banks), D + 32 for V (transposing reads bank-disjoint). INT8: each tile's key
// scales (times scale_log2) and value scales, in a four-tile ring (staged with the keys, two
// tiles ahead, and read by the softmax).
template <int D, bool INT8>
struct PPTiles {
    static constexpr int KROW = D + 8, VROW = D + 32;
    uint16_t k[2][KT * KROW];
    uint16_t v[2][KT * VROW];
    float s[INT8 ? 4 : 1][INT8 ? 2 * KT : 4];
};

__device__ __forceinline__ u32x2 lds_tr16(const uint16_t *p) {
    const s16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (__attribute__((address_space(3))) s16x4 *)(__attribute__((address_space(3))) uint16_t *)p);
    return __builtin_bit_cast(u32x2, v);
}

template <int I> using IC = std::integral_constant<int, I>;

// f(IC<0>{}), ..., f(IC<N - 1>{})
template <int N, int I = 0, typename F>
__device__ __forceinline__ void unroll(F &&f) {
    if constexpr (I < N) {
        f(IC<I>{});
        unroll<N, I + 1>(f);
    }
}

template <int D, bool INT8, int FORM>
__global__ void __launch_bounds__(FORM == TI_PP_SOLO ? 256 : 512, FORM == TI_PP_SOLO && D == 64 ? 3 : 2)
prefill_pp_kernel(PPParams p) {
    constexpr bool KS = FORM == TI_PP_KSPLIT, SOLO = FORM == TI_PP_SOLO;
    static_assert(D == 128 || KS || SOLO, "head_dim 64 stages a tile with one team");
    constexpr int NW = SOLO ? 4 : 8;
    constexpr int NQB = D / 16;        // score MFMAs per tile (16 head-dim elements each)
    constexpr int NDB = D / 32;        // 32-row blocks of O^T
    constexpr int RW = KS || SOLO ? 128 : 256; // packed query rows per work-group
    constexpr int GT = KS || SOLO ? 256 : 512; // threads that stage a tile
    constexpr int CPR = D / 8;         // 8-element chunks per row
    constexpr int NC = KT * CPR / GT;  // chunks of K and of V per thread and tile
    // Steps between a value chunk's load and its store into LDS (keys: 2). The 128-row form at
    // D = 128 stages two chunks per thread and has registers for one step's values only.
    constexpr int LV = D == 128 && GT == 256 ? 1 : 2;
    using Tiles = PPTiles<D, INT8>;
    using Chunk = std::conditional_t<INT8, u32x2, u32x4>;
    constexpr int KROW = Tiles::KROW, VROW = Tiles::VROW;
    constexpr int SLAB = KS ? NW * 64 * (NDB / 2 * 64 + 8) : 0;   // the merge's exchange area (bytes)
    constexpr int TILES = (KS ? 2 : 1) * (int)sizeof(Tiles);
    __shared__ __attribute__((aligned(16))) char smem_raw[TILES > SLAB ? TILES : SLAB];

    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int team = SOLO ? 0 : w >> 2;                       // 0: A, 1: B
    const int r32 = lane & 31, kg = lane >> 5;
    Tiles &sm = reinterpret_cast<Tiles *>(smem_raw)[KS ? team : 0];
    // Grid (Hk, q-tiles x splits, B): consecutive work-groups (dealt round-robin to the 8 XCDs)
    // belong to different KV heads, so each head's K/V stays in one XCD's L2.
    const int h = blockIdx.x, b = blockIdx.z;
    const int qt = p.qtiles - 1 - (int)(blockIdx.y >> p.sshift);   // heaviest q-tiles first
    const int split = (int)blockIdx.y & (p.splits - 1);
    // the pointer arguments the prologue dereferences, in the kernel arguments' first batch
    asm volatile("" ::"s"(p.bt), "s"(p.positions), "s"(p.qsl), "s"(p.kp), "s"(p.vp), "s"(p.q));
    const int32_t *bt = p.bt + (size_t)b * p.bt_stride;
    // This thread's staging chunks: key ckey + (GT / CPR) u, elements cch * 8 .. + 8. A wave's
    // chunk u lies in one 16-key half of the tile (half_of), so its row base is scalar.
    const int gt = tid % GT, ckey = gt / CPR, cch = gt % CPR;
    constexpr int KPU = GT / CPR;
    const int wave_half = __builtin_amdgcn_readfirstlane(ckey >> 4);
    auto half_of = [&](int u) { return NC == 2 ? u : wave_half; };
    const uint32_t chunk_off = (uint32_t)((ckey & 15) * D + cch * 8) * (INT8 ? 1 : 2);
    // Block-table entries of a tile's halves (raw: scalar loads, looked up a phase before use).
    // NH = 1: only this wave's half (its chunks lie in one, and there are no scales to find).
    constexpr int NH = NC == 2 || INT8 ? 2 : 1, EB = INT8 ? 1 : 2;
    struct Pages {
        int pg[NH];
    };
    auto half_pos = [&](int kt, int x) { return kt * KT + 16 * (NH == 2 ? x : wave_half); };
    auto pages_at = [&](int kt) {
        Pages r;
#pragma unroll
        for (int x = 0; x < NH; x++) r.pg[x] = sload(bt, min(half_pos(kt, x) >> p.pshift, p.bt_stride - 1));
        return r;
    };
    // Without key splits the first tiles' entries do not depend on the sequence's position:
    // their loads go out together with those of the query counts.
    Pages rp[4];
    auto first_pages = [&](int lo) {
#pragma unroll
        for (int j = 0; j < 4; j++) rp[j] = pages_at(KS ? lo + 2 * j + team : lo + j);
    };
    if (p.splits == 1) first_pages(0);
    const int tok0 = p.qsl ? sload(p.qsl, b) : b * p.nmax;
    const int nb = p.qsl ? min(sload(p.qsl, b + 1) - tok0, p.nmax) : p.nmax;   // at most max_query_len
    const int t_first = qt * p.TQ;
    if (t_first >= nb) return;
    const int start = max(sload(p.positions, tok0), 0), len = start + nb;   // a negative position reads as 0
    const int t_last = min(t_first + p.TQ, nb) - 1;
    const int kend = p.causal ? start + t_last + 1 : len;
    const int nkt = (kend + KT - 1) / KT;
    const int per = (nkt + p.splits - 1) / p.splits;
    const int kt_lo = min(split * per, nkt), kt_hi = min(kt_lo + per, nkt);
    const int N = KS ? (kt_hi - kt_lo + 1) / 2 : kt_hi - kt_lo;   // steps of this work-group
    const size_t unit = ((size_t)b * p.Hk + h) * p.splits + split;
    const int mask_from = p.causal ? start + t_first : len - 1;
    if (N == 0) {
        // A split with no keys: neutral partials (m = -big, l = 0, acc = 0).
        for (int idx = tid; idx < RW * (D + 2); idx += 64 * NW) {
            const int rr = idx / (D + 2), c = idx - rr * (D + 2);
            const int ttl = rr / p.G, gg = rr - ttl * p.G, tt = t_first + ttl;
            if (ttl < p.TQ && tt < nb)
                p.part[(unit * p.M + (size_t)tt * p.G + gg) * (D + 2) + c] = c == D ? NEG_BIG : 0.0f;
        }
        return;
    }

    // Key tile of step j (this team's, KS; its odd tile out is masked by position).
    auto tile = [&](int j) { return KS ? kt_lo + 2 * j + team : kt_lo + j; };

    // Row offsets of a tile's halves in bytes from the KV head's first row (page clamped into
    // the pool; an entry of 0 or less wraps and reads the last page). Tiles past the last are
    // loaded from whatever page the table's next entries name, never used.
    struct Bases {
        uint64_t e[NH];
    };
    const uint32_t pstride = (uint32_t)p.Hk * p.P * D * EB;
    const size_t hoff = (size_t)h * p.P * D * EB, half_q = (size_t)p.num_pages * p.Hk * p.P * D;
    const char *kbase = (INT8 ? (const char *)p.lq : (const char *)p.kp) + hoff;
    const char *vbase_g = INT8 ? kbase + half_q : (const char *)p.vp + hoff;
    auto bases = [&](const Pages &r, int j) {
        Bases o;
#pragma unroll
        for (int x = 0; x < NH; x++)
            o.e[x] = (uint64_t)min((uint32_t)(r.pg[x] - 1), (uint32_t)p.num_pages - 1) * pstride +
                     (uint32_t)((half_pos(tile(j), x) & (p.P - 1)) * (D * EB));
        return o;
    };
    auto base_of = [&](const Bases &o, int u) { return NH == 2 && half_of(u) ? o.e[NH - 1] : o.e[0]; };

    // a scalar base plus a per-lane 32-bit offset (scalar-base addressing)
    auto chunk_at = [&](const char *base, uint64_t off) {
        const uint64_t a = (uint64_t)base + off;
        const uint64_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)a);
        const uint64_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(a >> 32));
        typedef const __attribute__((address_space(1))) char *global_ptr;
        return *(const __attribute__((address_space(1))) Chunk *)((global_ptr)((hi << 32) | lo) + chunk_off);
    };
    const size_t half_s = (size_t)p.num_pages * p.Hk * p.P;
    Chunk sk[2][NC], sv[LV][NC];                   // staged chunks
    float ss[2];                                   // INT8: staged scale of key lane % 32 (keys', then values')
    auto load_k = [&](Chunk &r, const Bases &o, int u) { r = chunk_at(kbase, base_of(o, u)); };
    auto load_v = [&](Chunk &r, const Bases &o, int u) { r = chunk_at(vbase_g, base_of(o, u)); };
    const float *sbase = p.ls + (size_t)h * p.P + (kg ? half_s : 0) + (r32 & 15);
    auto load_s = [&](float &r, const Bases &o) {
        // every wave loads the same 64 scales (no branch: the count of loads in flight stays
        // static), one wave of the staging threads stores them
        r = sbase[(r32 >> 4 ? o.e[NH - 1] : o.e[0]) / D];
    };
    auto bf16_chunk = [&](const Chunk &r) -> u32x4 {
        if constexpr (INT8) {
            u32x4 o;
            uint32_t a, b2, c, d;
            i8x4_to_bf16(r[0], a, b2);
            i8x4_to_bf16(r[1], c, d);
            o[0] = a, o[1] = b2, o[2] = c, o[3] = d;
            return o;
        } else {
            return r;
        }
    };
    auto store_k = [&](const Chunk &r, int buf, int u) {
        *reinterpret_cast<u32x4 *>(&sm.k[buf][(ckey + KPU * u) * KROW + cch * 8]) = bf16_chunk(r);
    };
    auto store_v = [&](const Chunk &r, int buf, int j, int u) {
        // Keys past kend in the last tile may hold any bits (even NaN) of an allocated
        // page: their probabilities are 0 and their values must be finite. Branch-free,
        // so the stage registers are never rewritten while loads are pending.
        const uint32_t keep = tile(j) * KT + ckey + KPU * u < kend ? ~0u : 0u;
        *reinterpret_cast<u32x4 *>(&sm.v[buf][(ckey + KPU * u) * VROW + cch * 8]) = bf16_chunk(r) & keep;
    };
    const float smul = kg ? 1.0f : p.scale_log2;
    auto store_s = [&](float r, int j) {
        // scales of keys past kend may hold any bits too: zero
        if (w == (KS ? 4 * team : 0)) sm.s[j & 3][lane] = tile(j) * KT + r32 < kend ? r * smul : 0.0f;
    };

    // Query rows (B operand of S^T = K Q^T): wave w holds rows 32 w .. 32 w + 31 (KS: both
    // teams hold the same 128).
    const int r = (KS ? w & 3 : w) * 32 + r32, tl = r / p.G, g = r - tl * p.G, t = t_first + tl;
    const bool row_ok = tl < p.TQ && t < nb;
    // last visible key of the row (KS: of this split too, whose odd tile out is masked by it)
    const int qpos = min(p.causal && row_ok ? start + t : len - 1, kt_hi * KT - 1);

    // Prologue: K of tiles 0 and 1 in LDS; K of tiles 2, 3 and V of tiles 0 .. LV - 1 in
    // flight (in the order of their stores, so the waits before each store count exactly the
    // younger loads).
    Bases bs[4];                                   // bases of tiles i + 1 .. i + 3 in 1 .. 3
    Pages raw4;                                    // block-table entries of tile i + 4
    bf16x8 qreg[NQB];
    {
        if (p.splits != 1) first_pages(kt_lo);
#pragma unroll
        for (int j = 0; j < 4; j++) bs[j] = bases(rp[j], j);
        Chunk k0[NC], k1[NC];
        float s0 = 0.0f, s1 = 0.0f;
#pragma unroll
        for (int u = 0; u < NC; u++) load_k(k0[u], bs[0], u);
        if constexpr (INT8) load_s(s0, bs[0]);
#pragma unroll
        for (int u = 0; u < NC; u++) load_k(k1[u], bs[1], u);
        if constexpr (INT8) load_s(s1, bs[1]);
        __builtin_amdgcn_sched_barrier(0);
        const uint16_t *qr = p.q + ((size_t)(tok0 + (row_ok ? t : 0)) * p.Hq + h * p.G + (row_ok ? g : 0)) * D;
        u32x4 raw[NQB];
#pragma unroll
        for (int i = 0; i < NQB; i++) raw[i] = *reinterpret_cast<const u32x4 *>(qr + i * 16 + kg * 8);
#pragma unroll
        for (int x = 0; x < 2; x++) {
            __builtin_amdgcn_sched_barrier(0);
            if (x < LV) {
#pragma unroll
                for (int u = 0; u < NC; u++) load_v(sv[x % LV][u], bs[x], u);
            }
#pragma unroll
            for (int u = 0; u < NC; u++) load_k(sk[x][u], bs[2 + x], u);
            if constexpr (INT8) load_s(ss[x], bs[2 + x]);
        }
        __builtin_amdgcn_sched_barrier(0);
        raw4 = pages_at(tile(4));
#pragma unroll
        for (int u = 0; u < NC; u++) store_k(k0[u], 0, u);
        if constexpr (INT8) store_s(s0, 0);
#pragma unroll
        for (int u = 0; u < NC; u++) store_k(k1[u], 1, u);
        if constexpr (INT8) store_s(s1, 1);
        const uint32_t keep = row_ok ? ~0u : 0u;
#pragma unroll
        for (int i = 0; i < NQB; i++) {
            if constexpr (INT8) {
                // bf16(q * smooth) (attention.jl:90-95)
                const int d0 = i * 16 + kg * 8;
#pragma unroll
                for (int e = 0; e < 4; e++)
                    raw[i][e] = pack_bf16x2(__uint_as_float(raw[i][e] << 16) * p.smooth[d0 + 2 * e],
                                            __uint_as_float(raw[i][e] & 0xffff0000u) * p.smooth[d0 + 2 * e + 1]);
            }
            qreg[i] = as_bf16x8(raw[i] & keep);
        }
    }

    f32x16 o[NDB];
#pragma unroll
    for (int db = 0; db < NDB; db++)
#pragma unroll
        for (int e = 0; e < 16; e++) o[db][e] = 0.0f;
    float m = NEG_BIG, l = 0.0f;
    bf16x8 pb[2];
    pb[0] = pb[1] = as_bf16x8((u32x4){0u, 0u, 0u, 0u});
    f32x16 sc;

    const int c16 = lane >> 4, s16 = lane & 15;
    const int tr_row = 4 * (c16 >> 1) + (s16 >> 2), tr_col = 16 * (c16 & 1) + 4 * (s16 & 3);

    u32x4 ka[NQB];                     // K operands of the next score product
    u32x2 va[2 * NDB][2];              // V^T operands of the value product
    auto read_k = [&](int kb, int i) {
        ka[i] = *reinterpret_cast<const u32x4 *>(&sm.k[kb][r32 * KROW + kg * 8] + i * 16);
    };
    // value MFMA x: keys 16 (x / NDB) .. + 15, output block x % NDB
    auto read_v = [&](int vb, int x) {
        const uint16_t *vbase = &sm.v[vb][tr_row * VROW + tr_col] + 16 * (x / NDB) * VROW + 32 * (x % NDB);
        va[x][0] = lds_tr16(vbase);
        va[x][1] = lds_tr16(vbase + 8 * VROW);
    };
    auto pv = [&](int x) {
        o[x % NDB] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
            as_bf16x8((u32x4){va[x][0][0], va[x][0][1], va[x][1][0], va[x][1][1]}), pb[x / NDB], o[x % NDB], 0, 0, 0);
    };
    auto qk = [&](int i) {
        if (i == 0) {
#pragma unroll
            for (int e = 0; e < 16; e++) sc[e] = 0.0f;
        }
        sc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf16x8(ka[i]), qreg[i], sc, 0, 0, 0);
    };
    // Online softmax of step j's scores (exp2 domain, lazy rescale after the first p.eager steps)
    // -> pb. Only tiles reaching past mask_from (the diagonal / last tiles) compare key positions.
    const int jm = min(mask_from + 1, kt_hi * KT); // first key position that a row may not see
    auto softmax = [&](int j) {
        const int kt = tile(j);
        f32x4 svq[4];
        if constexpr (INT8) {
            // a lane's scores are of keys 8 (e / 4) + 4 kg + e % 4
            const float *sp = &sm.s[j & 3][4 * kg];
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const f32x4 skq = *reinterpret_cast<const f32x4 *>(sp + 8 * q);
                svq[q] = *reinterpret_cast<const f32x4 *>(sp + KT + 8 * q);
#pragma unroll
                for (int e = 0; e < 4; e++) sc[4 * q + e] *= skq[e];   // scaled to log2 units too
            }
        }
        if (kt * KT + KT > jm) {
            // A real branch (the empty asm keeps the compiler from if-converting the
            // selects into every tile): key 8 (e / 4) + 4 kg + e % 4 is visible iff
            // it is <= qpos - kt * KT.
            asm volatile("");
            const int lim = qpos - kt * KT - 4 * kg;
#pragma unroll
            for (int e = 0; e < 16; e++)
                sc[e] = 8 * (e >> 2) + (e & 3) <= lim ? sc[e] : -INFINITY;
        }
        float mt = -INFINITY;
#pragma unroll
        for (int e = 0; e < 16; e++) mt = fmaxf(mt, sc[e]);
        if constexpr (!INT8) mt *= p.scale_log2;
        if (__any(mt > m + (j < p.eager ? 0.0f : RESCALE_LOG2))) {
            mt = fmaxf(mt, __shfl_xor(mt, 32));
            const float mn = fmaxf(m, mt);
            const float alpha = fast_exp2(m - mn);
            m = mn;
            l *= alpha;
#pragma unroll
            for (int db = 0; db < NDB; db++) o[db] *= alpha;
        }
        float pe[16], ps = 0.0f;
#pragma unroll
        for (int e = 0; e < 16; e++) {
            pe[e] = fast_exp2(INT8 ? sc[e] - m : __builtin_fmaf(sc[e], p.scale_log2, -m));
            ps += pe[e];
            if constexpr (INT8) pe[e] *= svq[e >> 2][e & 3];
        }
        l += ps;
#pragma unroll
        for (int hh = 0; hh < 2; hh++)
            pb[hh] = as_bf16x8((u32x4){pack_bf16x2(pe[8 * hh + 0], pe[8 * hh + 1]), pack_bf16x2(pe[8 * hh + 2], pe[8 * hh + 3]),
                                       pack_bf16x2(pe[8 * hh + 4], pe[8 * hh + 5]), pack_bf16x2(pe[8 * hh + 6], pe[8 * hh + 7])});
    };

    // Phase boundary: no instruction is scheduled across it, so each phase keeps only its
    // own work (the matrix-core phase must not absorb softmax VALU work).
    auto phase_barrier = [] {
        __builtin_amdgcn_sched_barrier(0);
        __syncthreads();
        __builtin_amdgcn_sched_barrier(0);
    };
    // Phase X_i (S = i % 2; FIRST: i = 0, no values yet). MFMAs: three scores, then values and
    // scores in turn (independent accumulators), then the values left. The gaps between them
    // (32 cycles each, about five instructions) take the side operations: value operands of
    // tile i - 1; V(i) and K(i + 2) into LDS (loaded LV and 2 steps before); the offsets of
    // tile i + 4; the staging registers' next loads; key operands of tile i + 1 (a key
    // operand's register is free once its score MFMA has issued). gap_of: the MFMA after which
    // operation X is issued, for 16 MFMAs (D = 128), halved for D = 64.
    auto phase_x = [&](int i, auto slot, auto first) {
        constexpr int S = decltype(slot)::value, S1 = 1 - S, SV = S % LV;
        constexpr bool FIRST = decltype(first)::value;
        constexpr int NM = NQB + 2 * NDB, SC = INT8 ? 1 : 0;
        constexpr int O_SV = 2 * NDB, O_SK = O_SV + NC, O_SS = O_SK + NC, O_BA = O_SS + SC, O_LV = O_BA + NH,
                      O_LK = O_LV + NC, O_LS = O_LK + NC, O_RK = O_LS + SC, NS = O_RK + NQB;
        constexpr auto gap_of = [](int X) {
            const int g = X < O_SV   ? X * 8 / O_SV / 2
                          : X < O_SK ? 4 + (X - O_SV)
                          : X < O_SS ? (NC == 2 ? 6 : 5) + (X - O_SK)
                          : X < O_BA ? 7
                          : X < O_LV ? 7 + (X - O_BA)
                          : X < O_LK ? 8 + (X - O_LV)
                          : X < O_LS ? 9 + (X - O_LK)
                          : X < O_RK ? 11
                                     : 9 + (X - O_RK) * 8 / NQB / 2;
            return g * NM / 16;
        };
        Bases b4;
        unroll<NM>([&](auto mi) {
            constexpr int M = decltype(mi)::value;
            constexpr int T = M - 3;               // after the first three scores
            constexpr bool IS_QK = M < 3 || (T / 2 < NQB - 3 && T % 2 == 1);
            if constexpr (IS_QK) qk(M < 3 ? M : 3 + T / 2);
            else if constexpr (!FIRST) pv(T / 2 < NQB - 3 ? T / 2 : T - (NQB - 3));
            unroll<NS>([&](auto xi) {
                constexpr int X = decltype(xi)::value;
                if constexpr (gap_of(X) == M) {
                    if constexpr (X < O_SV) {
                        if constexpr (!FIRST) read_v(S1, X);
                    } else if constexpr (X < O_SK) {
                        store_v(sv[SV][X - O_SV], S, i, X - O_SV);
                    } else if constexpr (X < O_SS) {
                        store_k(sk[S][X - O_SK], S, X - O_SK);
                    } else if constexpr (X < O_BA) {
                        store_s(ss[S], i + 2);
                    } else if constexpr (X < O_LV) {
                        b4.e[X - O_BA] = bases(raw4, i + 4).e[X - O_BA];
                    } else if constexpr (X < O_LK) {
                        load_v(sv[SV][X - O_LV], bs[LV], X - O_LV);
                    } else if constexpr (X < O_LS) {
                        load_k(sk[S][X - O_LK], b4, X - O_LK);
                    } else if constexpr (X < O_RK) {
                        load_s(ss[S], b4);
                    } else {
                        read_k(S1, X - O_RK);
                    }
                }
            });
            __builtin_amdgcn_sched_barrier(0);
        });
        bs[1] = bs[2], bs[2] = bs[3], bs[3] = b4;
    };
    auto phase_y = [&](int i) {
        raw4 = pages_at(tile(i + 5));
        softmax(i);
        // the lookup's wait falls here, where the barrier waits for LDS anyway
        asm volatile("" : "+s"(raw4.pg[0]));
        if constexpr (NH == 2) asm volatile("" : "+s"(raw4.pg[NH - 1]));
    };

    phase_barrier();
#pragma unroll
    for (int q = 0; q < NQB; q++) read_k(0, q);
    phase_barrier();                               // X_0 overwrites tile 0's keys
    if (!SOLO && team == 1) phase_barrier();       // team B runs one phase behind
    // SOLO: one barrier a step
    auto x_barrier = [&] {
        if constexpr (!SOLO) phase_barrier();
        else __builtin_amdgcn_sched_barrier(0);
    };
    phase_x(0, IC<0>{}, std::true_type{});
    x_barrier();
    // Whole pairs of steps, then the last one or two: a loop with one exit keeps the count of
    // loads in flight static, so the waits before the LDS stores leave the younger ones pending.
    int i = 0;
    for (; i + 2 < N; i += 2) {
        phase_y(i);
        phase_barrier();
        phase_x(i + 1, IC<1>{}, std::false_type{});
        x_barrier();
        phase_y(i + 1);
        phase_barrier();
        phase_x(i + 2, IC<0>{}, std::false_type{});
        x_barrier();
    }
    phase_y(i);
    phase_barrier();
    if (i + 1 < N) {
        phase_x(i + 1, IC<1>{}, std::false_type{});
        x_barrier();
        phase_y(i + 1);
        phase_barrier();
    }
    // last tile's values
#pragma unroll
    for (int x = 0; x < 2 * NDB; x++) read_v((N - 1) & 1, x);
#pragma unroll
    for (int x = 0; x < 2 * NDB; x++) pv(x);
    if (!SOLO && team == 0) phase_barrier();

    l += __shfl_xor(l, 32);
    // The output blocks this wave writes: all of them, or (KS) half of them after the teams'
    // states are merged: each wave hands the other team's wave of its rows (same rows, same
    // lane layout) the half it does not write.
    int db0 = 0;
    constexpr int NOUT = KS ? NDB / 2 : NDB;
    if constexpr (KS) {
        f32x4 *slab = reinterpret_cast<f32x4 *>(smem_raw);
        float2 *ml = reinterpret_cast<float2 *>(smem_raw + NW * 64 * NOUT * 64);
        __syncthreads();                           // every wave is done with the tiles
        auto give = [&](int d0) {
#pragma unroll
            for (int x = 0; x < NOUT; x++)
#pragma unroll
                for (int e4 = 0; e4 < 4; e4++)
                    slab[(w * NOUT * 4 + 4 * x + e4) * 64 + lane] =
                        (f32x4){o[d0 + x][4 * e4], o[d0 + x][4 * e4 + 1], o[d0 + x][4 * e4 + 2], o[d0 + x][4 * e4 + 3]};
        };
        if (team == 0) give(NOUT);
        else give(0);
        ml[w * 64 + lane] = make_float2(m, l);
        __syncthreads();
        const int ow = w ^ 4;
        const float2 oml = ml[ow * 64 + lane];
        const float mx = fmaxf(m, oml.x), wa = fast_exp2(m - mx), wb = fast_exp2(oml.x - mx);
        auto take = [&](int d0) {
#pragma unroll
            for (int x = 0; x < NOUT; x++)
#pragma unroll
                for (int e4 = 0; e4 < 4; e4++) {
                    const f32x4 v = slab[(ow * NOUT * 4 + 4 * x + e4) * 64 + lane];
#pragma unroll
                    for (int e = 0; e < 4; e++) o[x][4 * e4 + e] = o[d0 + x][4 * e4 + e] * wa + v[e] * wb;
                }
        };
        if (team == 0) take(0);
        else take(NOUT);
        m = mx;
        l = l * wa + oml.y * wb;
        db0 = team * NOUT;
    }
    if (!row_ok) return;
    if (p.splits > 1) {
        float *dst = p.part + (unit * p.M + (size_t)t * p.G + g) * (D + 2);
#pragma unroll
        for (int db = 0; db < NOUT; db++)
#pragma unroll
            for (int e4 = 0; e4 < 4; e4++)
                *reinterpret_cast<f32x4 *>(dst + 32 * (db0 + db) + 8 * e4 + 4 * kg) =
                    (f32x4){o[db][4 * e4], o[db][4 * e4 + 1], o[db][4 * e4 + 2], o[db][4 * e4 + 3]};
        if (kg == 0 && db0 == 0) *reinterpret_cast<float2 *>(dst + D) = make_float2(m, l);
        return;
    }
    const float inv = 1.0f / l;
    uint16_t *orow = p.out + ((size_t)(tok0 + t) * p.Hq + h * p.G + g) * D;
#pragma unroll
    for (int db = 0; db < NOUT; db++)
#pragma unroll
        for (int e4 = 0; e4 < 4; e4++) {
            const int d = 32 * (db0 + db) + 8 * e4 + 4 * kg;
            const uint32_t w0 = pack_bf16x2(o[db][4 * e4 + 0] * inv, o[db][4 * e4 + 1] * inv);
            const uint32_t w1 = pack_bf16x2(o[db][4 * e4 + 2] * inv, o[db][4 * e4 + 3] * inv);
            *reinterpret_cast<u32x2 *>(orow + d) = (u32x2){w0, w1};
        }
}

template <int D, bool INT8, int FORM>
void launch_pp(const PPParams &p, int B, hipStream_t s) {
    prefill_pp_kernel<D, INT8, FORM><<<dim3(p.Hk, p.qtiles * p.splits, B), FORM == TI_PP_SOLO ? 256 : 512, 0, s>>>(p);
}

template <int D, bool INT8>
void launch_pp_form(const PPParams &p, int form, int B, hipStream_t s) {
    if constexpr (D == 128 && !INT8) {
        if (form == TI_PP_SHARED) return launch_pp<D, INT8, TI_PP_SHARED>(p, B, s);
    }
    if (form == TI_PP_SOLO) launch_pp<D, INT8, TI_PP_SOLO>(p, B, s);
    else launch_pp<D, INT8, TI_PP_KSPLIT>(p, B, s);
}

}  // namespace

// The ping-pong kernel takes bf16 activations over dense or INT8 caches with head_dim 64 or
// 128, power-of-two pages of at least 16 tokens (a page of all KV heads under 4 GiB: 32-bit
// strides) and at most 64 heads per KV head (as every prefill kernel).
//
// The library's pick counts the launch's 128-row work-groups, W; its 64-row ones, q64, the
// four-wave plan's on small launches; and the 32-key tiles that a block table has room for
// (nothing else on the host bounds the contexts). Head counts 32 / 8 unless stated; each figure:
// this form against the kernel that takes the step otherwise, the four-wave or the 16-row paired
// one, same process, graph replays, keys from HBM. A KSPLIT work-group has a CU to itself and
// costs about 7 us beside its steps (first loads, merge, stores), so it wins where those steps
// are many and loses where half its rows are padding or a second round is short.
//   W <= 128: none (512 tokens: the 16-row kernel's one round of 256 takes 9.3 us).
//   q64 < 256: none. From 32 tiles the four-wave plan's key splits even out ragged contexts (17 x
//     16 tokens on 500 to 4000: 46 us, KSPLIT 57); below, unsplit, it is the 16-row kernel (17 x
//     16 on 200 9.9, KSPLIT 11.3; 6 x 66 from scratch 7.8, 9.8). But KSPLIT from 32 to 40 tiles
//     (17 x 16 on 700 20.0 against 29.4), and from W = 192 (24 x 16 on 4096 80.5 against 99.3,
//     ragged to 4000 65 against 70; to 8000 120 against 115).
//   One q-tile of up to 64 rows per sequence: none for W < 512, the 16-row kernel's range (32 x
//     16 on 4096 KSPLIT 98.9 against 91.8, on 200 12.6 against 11.2; INT8 107 against 72, and at
//     64 x 16 SOLO 196 against 150, but with narrow tables 9.1 against 13.9 for 64 x 9). From there
//     SOLO (96 x 16 on 200 31.0 against 39.8).
//   INT8, D = 128, whose 64-row work-groups fit that range: none (20 x 40 on 1000 KSPLIT 64
//     against 42). Nor does INT8 for W <= 256, counted by the tokens that the sequences hold (5
//     prompts of 37 to 119 on 800 to 2800 68 against 50): converting tiles doubles the staging there.
//     But batches of 160 and narrow tables, which leave the contexts little room to differ, take KSPLIT
//     (5 x 121 from scratch 13.7 against 14.5, D = 64 9.7 against 13.8).
//     Beyond, with few idle rows and more than 40 tiles, KSPLIT (1500 on 4096 206 against 232; two
//     prompts of 520 23.9 against 22.6), but at D = 64 only alone (20 x 95 on 3000 142 against 130).
//   W <= 512: KSPLIT. At most two work-groups per CU, one resident at a time, each with half
//     the steps of an unsplit q-tile: 520 tokens 15.5 against 16.8 us, 1000 22.9 against 26.4,
//     2000 46.2 against 56.2; 600 on 4096 64.5 against 114.5; D = 64, 1000 16.0 against 21.5.
//     q-tiles with rows to spare start later (G = 3: 800 tokens, W = 160, 19.4 against 18.4),
//     D = 64 by the tokens held (5 chunks of 37 to 119 on 800 to 2800 31.3 against 29.1).
//     Below 32 tiles and past one round only sequences of more than 8 q-tiles (D = 64: 10) have the
//     steps (four of 138 to 403 14.5 against 16.3; 12 x 90 19.0, 18.0; D = 64 8 x 256 16.0, 14.9).
//   more: SHARED for dense D = 128 (half the loads and LDS stores per row): 3072 tokens 88.7
//     against 119.4 us, 8192 493 against 539; else SOLO, whose work-groups share a CU (two,
//     D = 64 three) and hide each other's fixed cost: INT8 3072 tokens 116.4 against 147.4,
//     D = 64 8192 309 against 394, eight D = 64 prompts of 100 to 2000 tokens 58.8 against
//     78.3. SOLO also takes dense D = 128 batches whose sequences are short in queries and keys (16
//     x 300 tokens 39.8 against 42.1 on SHARED, 16 x 512 71.9, 74.9) or mostly absent (a prompt of
//     2000 beside 16 tokens 56.5, 65.4): 256-row tiles there are padding or have few steps. Not
//     longer ones (SOLO, SHARED: 8 x 1024 102, 100; 8 x 2048 331, 306; 8 x 4096 1163, 1041; 16 x
//     512 on 4096 609, 534).
// Over 3757 shapes on either side of these lines, of up to 128 sequences, uniform and ragged, steps
// take 0.87 times as long in the mean as on the kernels that took them before this one had forms.
// Slower by more than 3 %: 14, mostly batches of W < 200 whose contexts are ragged, which the host
// cannot see (7 x 66 on 200 to 930 21.6 against 18.5; 5 x 110 on 1000 each 23.6 against 36.0).
int ti_pick_prefill_pp(const ti_attention_args *a, const ti_kv_cache *c, int path, bool bound_keys) {
    const int G = a->q_heads / c->kv_heads, P = c->page_size, D = c->head_dim;
    if (a->dtype != TI_BF16 || (D != 64 && D != 128) || P < 16 || (P & (P - 1)) || G > 64 ||
        2ull * c->kv_heads * P * D > 0xffffffffull)
        return TI_PP_NONE;
    const bool dense = c->kind == TI_KV_DENSE, dense128 = dense && D == 128;
    if (path == TI_PATH_PREFILL_PINGPONG && dense128 && 256 % G == 0) return TI_PP_SHARED;
    if (path != TI_PATH_AUTO && path != TI_PATH_PREFILL) return TI_PP_NONE;
    const long long pairs = (long long)c->kv_heads * a->num_seqs, n = a->max_query_len;
    const long long TQ = 128 / G, T = (n + TQ - 1) / TQ, q64 = (n + 64 / G - 1) / (64 / G) * pairs;
    // grids hold 65535 q-tiles: 256-row ones where those have been taken, none where not
    if (T > 65535) return dense128 && 256 % G == 0 ? TI_PP_SHARED : TI_PP_NONE;
    long long W = T * pairs;
    const long long tiles = bound_keys ? ((long long)a->block_table_stride * P + 31) / 32 : 1LL << 40;
    // Only here does the four-wave plan split keys, and only from 32 tiles: a workspace query
    // (unbounded tiles) that answers KSPLIT is right for narrower tables too.
    if (q64 < 256)
        return dense && (dense128 || T > 2) && tiles >= 32 && W >= (tiles <= 40 ? 129 : 192) ? TI_PP_KSPLIT : TI_PP_NONE;
    const bool int8_128 = !dense && D == 128;
    if (T == 1 && q64 == W && W < (int8_128 && tiles >= 32 ? 513 : 512)) return TI_PP_NONE;
    if (int8_128 && W > 256 && W < 512 && q64 <= 512) return TI_PP_NONE;
    if (T <= 2 && W >= 512) return TI_PP_SOLO;
    if (tiles < 32 && W > 256 && W <= 512 && (T > 1 || !dense) && T <= (D == 64 ? 10 : 8)) return TI_PP_NONE;
    if (T <= 2) return D == 128 && W >= (dense ? 129 : 256) ? TI_PP_KSPLIT : TI_PP_NONE;
    const long long held = W * a->total_tokens / (n * a->num_seqs);
    if (!dense) {
        if (a->num_seqs > 1 && tiles < 32 && W < 256 && held >= 160) return TI_PP_KSPLIT;
        if (W <= 512 || (W <= 640 && tiles > 40)) W = held;
        if (W < (D == 64 && a->num_seqs == 1 ? 256 : 257)) return TI_PP_NONE;
        if (W > 512) return TI_PP_SOLO;
        return tiles > 40 && (D == 128 || a->num_seqs == 1) ? TI_PP_KSPLIT : TI_PP_NONE;
    }
    if ((D == 64 && W <= 512 ? held : W) < (128 % G == 0 ? 129 : tiles <= 40 ? 176 : 160)) return TI_PP_NONE;
    if (W <= 512) return TI_PP_KSPLIT;
    const bool padded = a->num_seqs >= 8 && W > 1024 && ((T <= 24 && tiles <= 40) || 4 * held < W);
    return dense128 && T > 6 && !padded ? TI_PP_SHARED : TI_PP_SOLO;
}

int ti_launch_prefill_pp(const ti_attention_args *a, const ti_kv_cache *c, const ti_prefill_plan &pl,
                         hipStream_t s) {
    PPParams p;
    p.q = (const uint16_t *)a->q;
    p.out = (uint16_t *)a->out;
    p.kp = (const uint16_t *)c->k_pages;
    p.vp = (const uint16_t *)c->v_pages;
    p.lq = c->layer_q;
    p.ls = c->layer_scale;
    p.smooth = c->smooth;
    p.positions = a->positions;
    p.qsl = a->query_start_loc;
    p.bt = a->block_tables;
    p.bt_stride = a->block_table_stride;
    p.num_pages = c->num_pages;
    p.P = c->page_size;
    p.pshift = __builtin_ctz(c->page_size);
    p.Hk = c->kv_heads;
    p.Hq = a->q_heads;
    p.G = a->q_heads / c->kv_heads;
    p.nmax = a->max_query_len;
    p.causal = a->causal;
    p.scale_log2 = a->scale * LOG2E;
    p.part = (float *)a->workspace;
    p.splits = pl.splits;
    p.sshift = __builtin_ctz(pl.splits);
    // Every key group's first maximum is a probability of exactly 1, so fewer groups round more on
    // short contexts. Where the kernels that this one replaces have more groups than the form (four
    // on 16-row waves and 64-row tiles, eight where they split blocks; two below 1024 work-groups
    // of 128 rows), its first steps rescale to every larger maximum, which brings the error against
    // 64 bits to theirs: 600 tokens 0.00196 (KSPLIT without 0.00200, the 16-row kernel 0.00196) for
    // 16.1 -> 16.5 us, 24 x 16 on 2000 0.00230 (0.00234, 0.00231) for 45.1 -> 45.4 (on 4096 77.0 ->
    // 80.5), five of 512 at head_dim 64 0.00198 (SOLO without 0.00204, four-wave 0.00200) for 20.8
    // -> 21.3.
    const long long T = (a->max_query_len + 128 / p.G - 1) / (128 / p.G), W = T * p.Hk * a->num_seqs;
    const bool dense128 = c->kind == TI_KV_DENSE && c->head_dim == 128;
    if (pl.pp == TI_PP_KSPLIT) p.eager = W > 256 ? 0 : T == 1 ? 8 : 3;
    else p.eager = W < 1024 && !(T == 1 && dense128) && a->path != TI_PATH_PREFILL_PINGPONG ? 4 : 0;
    p.M = pl.rows;
    p.TQ = pl.TQ;
    p.qtiles = pl.qtiles;
    const bool int8 = c->kind == TI_KV_INT8;
    if (c->head_dim == 64) {
        if (int8) launch_pp_form<64, true>(p, pl.pp, a->num_seqs, s);
        else launch_pp_form<64, false>(p, pl.pp, a->num_seqs, s);
    } else {
        if (int8) launch_pp_form<128, true>(p, pl.pp, a->num_seqs, s);
        else launch_pp_form<128, false>(p, pl.pp, a->num_seqs, s);
    }
    if (hipGetLastError() != hipSuccess) return TI_ERR_LAUNCH;
    return pl.splits > 1 ? ti_launch_combine(a, c, pl.rows, pl.splits, s) : TI_OK;
}
