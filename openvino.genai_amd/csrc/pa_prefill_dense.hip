// Chunked-prefill PagedAttention on the gfx950 matrix cores for dense chunks, head size 128, whose KV blocks go straight from
// global memory into LDS: 16-bit caches of the query's type, and u8 caches whose rows were widened to f16 integers
// beforehand (`pa_widen_kernel`, below).  Work items, arithmetic and precision are those of pa_prefill16.hip (S^T = K . Q^T, online
// softmax in the log2 domain, O^T += V^T . P^T with the probabilities as high and low halves).
//
// A 256-thread workgroup takes 128 query rows, 32 per wave; two workgroups share a CU (four K and four V slots each).  What a
// block of 32 tokens costs a wave: 48 matrix instructions (16 QK, 32 PV; 768 cycles of the matrix pipe) and some 110 vector
// instructions.  While another wave's matrix instructions fill the pipe, a wave issues a vector instruction every 8
// cycles (two per 16 x 16 x 32 product; transcendental and dot instructions take 12): neither unit has much room, and scalar
// instructions and branches cost a wave as much as vector ones.  Hence
//   * rows are looked up per lane, in an LDS table of the range's cache blocks: no scalar address arithmetic in the walk;
//   * whether a row's running maximum must be raised is asked lane by lane, the maximum over a row's lanes formed only then;
//   * S^T of block j and O^T of block j - 1 are one run of matrix instructions, the softmax of block j follows them.
// us per launch and layer, before (copies with scalar addresses and the row maximum per block; u8: codes widened by every
// workgroup on their way to LDS) / now: bf16 28 / 4 heads 2048 tokens behind 30000 1386 / 1330 (0.91 TF of products, 1.36 with the
// low halves, 1.02 PFLOP/s; 3 - 5 % by card, as a step 1381 / 1311 to 1422 / 1381), f16 32 / 8 heads 1024 behind 8000 222 / 203; u8 32 / 8 heads 6143 tokens 700 / 558 in a kernel
// trace, their rows widened in 8.
// Also tried here: 32 x 32 x 16 products (5.7 cycles per vector instruction beside them, but loads and copies of another wave do
// not issue at all while one is in flight), 512-thread workgroups whose halves alternate between matrix and vector work (the
// phases fit, the clock does not: 8 % fewer cycles in the same time).
#include "pa_prefill.h"

#include <climits>
#include <type_traits>

namespace pa {
namespace {

constexpr int HD = 128;             // head size
constexpr int ROWB = HD * 2;        // bytes of a row in LDS, in a 16-bit cache and of a widened row
constexpr int TILEB = TOK * ROWB;   // bytes of a (block, kv head) of K or V
constexpr int CPR = ROWB / 16;      // 16-byte pieces per row
constexpr int KS = HD / 32;         // k-steps of QK
constexpr int RT = HD / 16;         // 16-channel tiles of PV
constexpr int NW = 4;               // waves
constexpr int NG = 2;               // 16-row groups per wave
static_assert(16 * NG * NW == PREFILL_ROWS, "rows of a work item");
constexpr int MAX_RANGE = 128;      // KV blocks an item walks at most
constexpr int HDRB = 4 * TOK * 4;   // header bytes of a widened (block, kv head)

__device__ __forceinline__ void dma4(const uint8_t* src, uint8_t* lds_dst) {  // (see dma16: 64 x 4 bytes)
    typedef __attribute__((address_space(3))) void* lds_p;
    typedef const __attribute__((address_space(1))) void* glb_p;
    __builtin_amdgcn_global_load_lds((glb_p)src, (lds_p)lds_dst, 4, 0, 0);
}

template <int DT, int QDT, bool U8>
__global__ __launch_bounds__(64 * NW, 2) void pa_prefill_dense_kernel(PrefillArgs a) {
    static_assert(!U8 || DT == DT_F16, "u8 codes are multiplied as f16");
    static_assert(U8 || DT == QDT, "16-bit caches are used in the query's type");
    // (every slot an LDS object of its own: the compiler orders operand reads behind the copies that may write what they read)
    __shared__ __align__(16) uint8_t k0[TILEB], k1[TILEB], k2[TILEB], k3[TILEB];
    __shared__ __align__(16) uint8_t v0[TILEB], v1[TILEB], v2[TILEB], v3[TILEB];
    __shared__ uint32_t first_row[2 * MAX_RANGE];
    __shared__ __align__(16) uint8_t h0[U8 ? HDRB : 16], h1[U8 ? HDRB : 16], h2[U8 ? HDRB : 16], h3[U8 ? HDRB : 16];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 15, g = lane >> 4;
    const StepDev& st = a.st;
    const int Hq = a.sh.Hq, Hkv = a.sh.Hkv, G = a.G;
    const int hkv = blockIdx.x % Hkv;
    const PrefillItem item = a.items[blockIdx.x / Hkv];
    const int b = item.b;
    const int t0 = st.subsequence_begins[b];
    const int past = st.past_lens[b];
    const int q0 = item.q0;
    const int R = item.nq * G;  // query rows of this tile
    const int tb = item.tb, te = item.te, cnt = te - tb;
    const int sw = st.sliding_window;
    const int kv_len = past + st.subsequence_begins[b + 1] - t0;

    int row_pos[NG];  // global position of the row's token (-1: no such row)
    int row_id[NG];   // token * Hq + head
    s8v qreg[NG][KS];
#pragma unroll
    for (int gi = 0; gi < NG; ++gi) {
        // rows beyond R repeat the tile's last row; nothing of theirs is stored
        const bool ok = 32 * wv + 16 * gi + n < R;
        const int rho = min(32 * wv + 16 * gi + n, R - 1);
        const int qtok = q0 + rho / G;
        row_pos[gi] = ok ? past + qtok : -1;
        row_id[gi] = (t0 + qtok) * Hq + hkv * G + rho % G;
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            u4v v = *reinterpret_cast<const u4v*>(a.query + (long)row_id[gi] * HD + 32 * s + 8 * g);
            if (QDT != DT) {  // bf16 query against f16 operands
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    v[e] = pack2<DT_F16>(__builtin_bit_cast(float, v[e] << 16), __builtin_bit_cast(float, v[e] & 0xffff0000u));
            }
            qreg[gi][s] = __builtin_bit_cast(s8v, v);
        }
    }
    const float scl = st.scale * LOG2E;
    float qsum[NG] = {0.0f, 0.0f};  // u8: sum of the row's query elements (the headers carry the scale)
    if (U8) {
#pragma unroll
        for (int gi = 0; gi < NG; ++gi) {
            float part = 0.0f;
#pragma unroll
            for (int s = 0; s < KS; ++s) {
                const h8 qh = __builtin_bit_cast(h8, qreg[gi][s]);
#pragma unroll
                for (int e = 0; e < 8; ++e) part += (float)qh[e];
            }
            qsum[gi] = xor_sum_g(part);
        }
    }
    // steps whose block every row of this wave sees all of need no mask: free_j .. free_j + free_n
    int free_j;
    uint32_t free_n;
    {
        // rows that do not exist (beyond R) are left out: what they compute is never stored
        int lim = INT_MAX, low = INT_MIN;
#pragma unroll
        for (int gi = 0; gi < NG; ++gi) {
            lim = min(lim, row_pos[gi] < 0 ? INT_MAX : row_pos[gi]);
            low = max(low, row_pos[gi] + 1 - sw);
        }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            lim = min(lim, __shfl_xor(lim, o, WAVE));
            low = max(low, __shfl_xor(low, o, WAVE));
        }
        const int hi = __builtin_amdgcn_readfirstlane(lim), lo = sw > 0 ? __builtin_amdgcn_readfirstlane(max(low, 0)) : 0;
        const int first = max((lo + TOK - 1) / TOK - tb, 0), last = (hi == INT_MAX ? INT_MAX / TOK : (hi + 1) / TOK) - 1 - tb;
        free_j = last >= first ? first : INT_MAX;
        free_n = last >= first ? last - first : 0;
    }

    // the running maximum is kept negated (NO_MAX while the row has seen nothing), ready for the exponent's multiply-add
    constexpr float NO_MAX = 1e30f;
    float neg_m[NG] = {NO_MAX, NO_MAX}, lo_at[NG] = {-INFINITY, -INFINITY}, l_part[NG] = {0.0f, 0.0f}, zsum[NG] = {0.0f, 0.0f};
    f4 acc[NG][RT], sc[NG][2];
#pragma unroll
    for (int gi = 0; gi < NG; ++gi)
#pragma unroll
        for (int r = 0; r < RT; ++r) acc[gi][r] = f4{0.0f, 0.0f, 0.0f, 0.0f};
    u4v pb[NG], pl[NG];  // probabilities (u8: weights) of the block in work, high and low halves
    bool lo = true;      // ... whether the low halves are needed

    // ---- copies: wave w moves rows 8 w .. 8 w + 7 of a block in two instructions per tensor, lane l the piece that belongs at
    // LDS position l % 16 of row 8 w + l / 16 (+ 4): piece (l % 16) ^ (row & 15) of K, (l % 16) ^ 2 (row & 7) of V (operand reads
    // free of bank conflicts).  Where a row lies is looked up per lane, in an LDS table of the range's cache blocks.  Positions
    // beyond the last one repeat it: no row behind the sequence's tokens is read.
    const int bsz = U8 ? TOK : a.sh.bs, shift = 31 - __builtin_clz(bsz);
    const int blk0 = (tb * TOK) >> shift;
    const int last_rel = (U8 ? te * TOK : min(kv_len, te * TOK)) - 1 - (blk0 << shift);  // (widened rows behind the tokens are zeros)
    const long wide0 = U8 ? (long)a.wide_tile0[b] : 0;
    {
        const int32_t* table = a.block_indices + st.block_indices_begins[b] + blk0;
        for (int i = tid; i <= last_rel >> shift; i += 64 * NW)
            first_row[i] = U8 ? (uint32_t)(((wide0 + tb + i) * Hkv + hkv) * TOK) : ((uint32_t)table[i] * Hkv + hkv) * bsz;
    }
    const int my_row = 8 * wv + (lane >> 4), rel0 = tb * TOK - (blk0 << shift) + my_row;
    const uint8_t* const k_src = a.key_cache;
    const uint8_t* const v_src = a.value_cache;
    const uint32_t k_off0 = ((lane & 15) ^ (my_row & 15)) << 4, k_off1 = ((lane & 15) ^ ((my_row + 4) & 15)) << 4;
    const uint32_t v_off0 = ((lane & 15) ^ ((my_row & 7) << 1)) << 4, v_off1 = ((lane & 15) ^ (((my_row + 4) & 7) << 1)) << 4;
    struct Rows { uint32_t a, b; };
    auto row_of = [&](int j) __attribute__((always_inline)) {
        const int rel = min(rel0 + j * TOK, last_rel), more = min(rel0 + j * TOK + 4, last_rel) - rel;
        const uint32_t r = first_row[rel >> shift] + (uint32_t)(rel & (bsz - 1));
        return Rows{r, r + more};
    };
    auto copy_k = [&](const Rows& r, uint8_t* slot) __attribute__((always_inline)) {
        dma16(k_src + ((uint64_t)r.a * ROWB + k_off0), slot + wv * 2048);
        dma16(k_src + ((uint64_t)r.b * ROWB + k_off1), slot + wv * 2048 + 1024);
    };
    auto copy_v = [&](const Rows& r, uint8_t* slot) __attribute__((always_inline)) {
        dma16(v_src + ((uint64_t)r.a * ROWB + v_off0), slot + wv * 2048);
        dma16(v_src + ((uint64_t)r.b * ROWB + v_off1), slot + wv * 2048 + 1024);
    };
    // (headers: the even waves move the first half, the odd ones the second, each the same bytes)
    const uint8_t* const h_src = U8 ? reinterpret_cast<const uint8_t*>(a.wide_hdr) + ((wide0 + tb) * Hkv + hkv) * HDRB + (wv & 1) * 256 + lane * 4 : nullptr;
    auto copy_h = [&](int j, uint8_t* slot) __attribute__((always_inline)) {
        if constexpr (U8) dma4(h_src + (uint64_t)(uint32_t)min(j, cnt - 1) * (uint32_t)(Hkv * HDRB), slot + (wv & 1) * 256);
    };

    // ---- the matrix products -------------------------------------------------------------------------------------------
    // Byte offsets of this lane's operands within a slot: of K's k-step s `k_lane ^ (s << 6)` (and 16 rows further on), of V's
    // channel tile r `v_lane ^ (r << 5)`.  Opaque in each step: as loop invariants they would be added to the address of every
    // slot ahead of the loop, some sixty registers' worth.
    uint32_t k_lane = n * ROWB + ((g ^ n) << 4);
    uint32_t v_lane = (4 * g + (n >> 2)) * ROWB + (((n & 3) >> 1 ^ ((4 * g + (n >> 2)) & 7) << 1) << 4) + 8 * (n & 1);
    auto qk = [&](const uint8_t* kb) __attribute__((always_inline)) {
        asm volatile("" : "+v"(k_lane));
#pragma unroll
        for (int gi = 0; gi < NG; ++gi) sc[gi][0] = sc[gi][1] = f4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int s = 0; s < KS; ++s)
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const s8v kop = *reinterpret_cast<const s8v*>(kb + (k_lane ^ (s << 6)) + 16 * u * ROWB);
#pragma unroll
                for (int gi = 0; gi < NG; ++gi) sc[gi][u] = mma<DT>(kop, qreg[gi][s], sc[gi][u]);
            }
    };
    // V operands come through the LDS transpose read: source lane (e = n >> 2, q = n & 3) of a 16-lane group supplies 4
    // channels of token 16 h + 4 g + e; lane n receives channel 16 r + n of tokens 16 h + 4 g + 0..3
    auto load_v = [&](const uint8_t* vb, int r) __attribute__((always_inline)) {
        const uint8_t* p0 = vb + (v_lane ^ (r << 5));
        const s4v x = lds_read_tr16(p0), y = lds_read_tr16(p0 + 16 * ROWB);
        return s8v{x[0], x[1], x[2], x[3], y[0], y[1], y[2], y[3]};
    };
    constexpr bool LO_ALWAYS = U8 || DT == DT_BF16;
    auto pv = [&](const uint8_t* vb) __attribute__((always_inline)) {
        asm volatile("" : "+v"(v_lane));
        if constexpr (LO_ALWAYS) {  // (a matrix instruction's result is ready some slots later: the low halves follow two tiles behind)
            s8v vop[RT];
#pragma unroll
            for (int r = 0; r < RT + 2; ++r) {
                if (r < RT) {
                    vop[r] = load_v(vb, r);
#pragma unroll
                    for (int gi = 0; gi < NG; ++gi) acc[gi][r] = mma<DT>(vop[r], __builtin_bit_cast(s8v, pb[gi]), acc[gi][r]);
                }
                if (r >= 2) {
#pragma unroll
                    for (int gi = 0; gi < NG; ++gi) acc[gi][r - 2] = mma<DT>(vop[r - 2], __builtin_bit_cast(s8v, pl[gi]), acc[gi][r - 2]);
                }
            }
        } else {
            auto half = [&](const u4v (&pp)[NG]) __attribute__((always_inline)) {
#pragma unroll
                for (int r = 0; r < RT; ++r) {
                    const s8v vop = load_v(vb, r);
#pragma unroll
                    for (int gi = 0; gi < NG; ++gi) acc[gi][r] = mma<DT>(vop, __builtin_bit_cast(s8v, pp[gi]), acc[gi][r]);
                }
            };
            half(pb);
            if (lo) half(pl);
        }
    };

    // ---- the softmax -------------------------------------------------------------------------------------------
    // The running maximum is only raised when a block exceeds it by more than 2^4: probabilities then stay below 16 and the
    // accumulators are rescaled a few times per row.  Whether any row of the wave has to be is asked lane by lane; the
    // maximum over a row's four lanes is formed only then.
    auto raise_to = [&](int gi, float mx, float& d) __attribute__((always_inline)) {  // mx: the block's maximum of the row (log2 domain)
        const float m_old = -neg_m[gi];
        const float m_new = mx + neg_m[gi] > 4.0f ? mx : m_old;
        d = m_old - m_new;  // 0 for a row that stays; -NO_MAX for one that held nothing (zeros)
        const float corr = __builtin_amdgcn_exp2f(d);
#pragma unroll
        for (int r = 0; r < RT; ++r) acc[gi][r] *= corr;
        l_part[gi] *= corr;
        zsum[gi] *= corr;
        neg_m[gi] = -m_new;
    };
    auto masked = [&](int gi, int tile, int jj, float x) __attribute__((always_inline)) {
        const int lim = row_pos[gi], low = sw > 0 ? max(0, lim + 1 - sw) : 0;
        const int pos = tile * TOK + 4 * g + 16 * (jj >> 2) + (jj & 3);
        return pos <= lim && pos >= low ? x : -INFINITY;
    };
    auto max8 = [](const float (&x)[8]) __attribute__((always_inline)) {
        return fmaxf(fmaxf(fmaxf(x[0], fmaxf(x[1], x[2])), fmaxf(x[3], x[4])), fmaxf(x[5], fmaxf(x[6], x[7])));
    };
    // 16-bit caches: see pa_prefill16.hip for the share from which the low halves of f16 probabilities are needed
    constexpr float LO_SHARE_LOG2 = -2.0f;
    // (the mask in a branch of its own: with two copies of all that follows the accumulators would be copied at their join)
    auto softmax16 = [&](bool edge, int tile) __attribute__((always_inline)) {
        float mx[NG];
        bool raise = false;
        if (edge) {
#pragma unroll
            for (int gi = 0; gi < NG; ++gi)
#pragma unroll
                for (int jj = 0; jj < 8; ++jj) sc[gi][jj >> 2][jj & 3] = masked(gi, tile, jj, sc[gi][jj >> 2][jj & 3]);
        }
#pragma unroll
        for (int gi = 0; gi < NG; ++gi) {
            float x[8];
#pragma unroll
            for (int jj = 0; jj < 8; ++jj) x[jj] = sc[gi][jj >> 2][jj & 3];
            mx[gi] = max8(x) * scl;
            raise |= mx[gi] + neg_m[gi] > 4.0f;
        }
        if (__any(raise)) {
#pragma unroll
            for (int gi = 0; gi < NG; ++gi) {
                float d;
                raise_to(gi, xor_max_g(mx[gi]), d);
                lo_at[gi] += d;
            }
        }
        bool need = false;
        float p[NG][8];
#pragma unroll
        for (int gi = 0; gi < NG; ++gi) {
#pragma unroll
            for (int jj = 0; jj < 8; ++jj) p[gi][jj] = __builtin_amdgcn_exp2f(fmaf(sc[gi][jj >> 2][jj & 3], scl, neg_m[gi]));
#pragma unroll
            for (int jj = 0; jj < 4; ++jj) {
                uint32_t hi = pack2<DT>(p[gi][2 * jj], p[gi][2 * jj + 1]);
                if (DT == DT_BF16) asm("" : "+v"(hi));  // (its halves are taken from this word, not converted once more)
                pb[gi][jj] = hi;
                if (LO_ALWAYS) l_part[gi] += p[gi][2 * jj] + p[gi][2 * jj + 1];  // (both halves follow: they hold it to 2^-17)
                else l_part[gi] = add_pair<DT>(hi, l_part[gi]);
            }
            need |= mx[gi] + neg_m[gi] > lo_at[gi];
        }
        if constexpr (!LO_ALWAYS) {
            lo = __any(need);
            if (lo) {
                // some row's largest probability is above the share of the denominator it was last compared with: look at the
                // denominators as they are now (this block included)
                need = false;
#pragma unroll
                for (int gi = 0; gi < NG; ++gi) {
                    lo_at[gi] = __log2f(xor_sum_g(l_part[gi])) + LO_SHARE_LOG2;
                    need |= mx[gi] + neg_m[gi] > lo_at[gi];
                }
                lo = __any(need);
            }
        }
        if (LO_ALWAYS || lo) {  // what the rounding dropped, as operands of their own (and into the denominator)
#pragma unroll
            for (int gi = 0; gi < NG; ++gi)
#pragma unroll
                for (int jj = 0; jj < 4; ++jj) {
                    const uint32_t hi = pb[gi][jj];
                    uint32_t low;
                    if (DT == DT_BF16) {
                        low = pack2<DT>(p[gi][2 * jj] - __builtin_bit_cast(float, hi << 16),
                                        p[gi][2 * jj + 1] - __builtin_bit_cast(float, hi & 0xffff0000u));
                    } else {
                        low = residual_f16x2(hi, p[gi][2 * jj], p[gi][2 * jj + 1]);
                    }
                    pl[gi][jj] = low;
                    if (!LO_ALWAYS) l_part[gi] = add_pair<DT>(low, l_part[gi]);
                }
        }
    };
    // u8 caches: headers hold, per token, K scale x logit scale | -(zero-point left of K) x that | V scale | zero-point left of V
    auto softmax_u8 = [&](bool edge, int tile, const uint8_t* hb) __attribute__((always_inline)) {
        const float* hdr = reinterpret_cast<const float*>(hb) + 4 * g;
        f4 sck[2], zpk[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            sck[u] = *reinterpret_cast<const f4*>(hdr + 16 * u);
            zpk[u] = *reinterpret_cast<const f4*>(hdr + TOK + 16 * u);
        }
        float x[NG][8];  // logits (log2 domain) less the running maximum
        bool raise = false;
#pragma unroll
        for (int gi = 0; gi < NG; ++gi)
#pragma unroll
            for (int jj = 0; jj < 8; ++jj)
                x[gi][jj] = fmaf(sc[gi][jj >> 2][jj & 3], sck[jj >> 2][jj & 3], fmaf(zpk[jj >> 2][jj & 3], qsum[gi], neg_m[gi]));
        if (edge) {
#pragma unroll
            for (int gi = 0; gi < NG; ++gi)
#pragma unroll
                for (int jj = 0; jj < 8; ++jj) x[gi][jj] = masked(gi, tile, jj, x[gi][jj]);
        }
#pragma unroll
        for (int gi = 0; gi < NG; ++gi) raise |= max8(x[gi]) > 4.0f;
        if (__any(raise)) {
#pragma unroll
            for (int gi = 0; gi < NG; ++gi) {
#pragma unroll
                for (int jj = 0; jj < 8; ++jj) {  // (anew: a logit less NO_MAX holds nothing of the logit)
                    x[gi][jj] = fmaf(sc[gi][jj >> 2][jj & 3], sck[jj >> 2][jj & 3], zpk[jj >> 2][jj & 3] * qsum[gi]);
                    if (edge) x[gi][jj] = masked(gi, tile, jj, x[gi][jj]);
                }
                float d;
                raise_to(gi, xor_max_g(max8(x[gi])), d);
#pragma unroll
                for (int jj = 0; jj < 8; ++jj) x[gi][jj] += neg_m[gi];
            }
        }
        f4 scv[2], zpv[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            scv[u] = *reinterpret_cast<const f4*>(hdr + 2 * TOK + 16 * u);
            zpv[u] = *reinterpret_cast<const f4*>(hdr + 3 * TOK + 16 * u);
        }
#pragma unroll
        for (int gi = 0; gi < NG; ++gi) {
            float p[8], psum = 0.0f, zs = 0.0f;
#pragma unroll
            for (int jj = 0; jj < 8; ++jj) {
                p[jj] = __builtin_amdgcn_exp2f(x[gi][jj]);
                psum += p[jj];
            }
#pragma unroll
            for (int jj = 0; jj < 4; ++jj) {
                typedef _Float16 h2 __attribute__((ext_vector_type(2)));
                const float w0 = p[2 * jj] * scv[jj >> 1][(2 * jj) & 3];
                const float w1 = p[2 * jj + 1] * scv[jj >> 1][(2 * jj + 1) & 3];
                uint32_t wb = __builtin_bit_cast(uint32_t, h2{(_Float16)w0, (_Float16)w1});
                asm volatile("" : "+v"(wb));  // one rounded value for both uses (see pa_prefill16.hip)
                pb[gi][jj] = wb;
                pl[gi][jj] = residual_f16x2(wb, w0, w1);
                zs = fmaf(w0, zpv[jj >> 1][(2 * jj) & 3], zs);
                zs = fmaf(w1, zpv[jj >> 1][(2 * jj + 1) & 3], zs);
            }
            l_part[gi] += psum;
            zsum[gi] += zs;
        }
    };
    auto softmax = [&](int j, const uint8_t* hb) __attribute__((always_inline)) {
        const int tile = tb + j;
        const bool edge = (uint32_t)(j - free_j) > free_n;  // wave-uniform
        if constexpr (U8) softmax_u8(edge, tile, hb);
        else softmax16(edge, tile);
    };

    // ---- the walk -----------------------------------------------------------------------------------------------
    // Step j: barrier | copies of later blocks go out | S^T of block j, O^T of block j - 1 | the wave's share of what step j + 1
    // reads has landed | softmax of block j.  Block j lives in slot j % 4 of K, V and (u8) headers.
    // Slots: step j copies K of block j + 3 over block j - 1, V of j + 2 and headers of j + 2 over j - 2: what was read from there was
    // read in step j - 1 at the latest, in front of this step's barrier.
    // Waits: a wave's copies land in order; at the end of step j only its newest COPIES may be outstanding, those of this step, so
    // that K up to block j + 2, V and headers up to j + 1 are there.  This is only right while a step issues exactly this many
    // copies and nothing else that counts (the build fails on spills, whose scratch traffic would).
    constexpr int COPIES_PER_TENSOR = TILEB / (NW * 64 * 16);  // dma16 moves 64 x 16 bytes
    static_assert(COPIES_PER_TENSOR == 2 && HDRB == 2 * 64 * 4, "copy_k and copy_v issue two copies each, copy_h one");
    constexpr int COPIES = 2 * COPIES_PER_TENSOR + (U8 ? 1 : 0);
    // The rows of a sequence's last block that lie behind its tokens repeat the last row; in V they are cleared, each wave its own
    // once they have landed: 0 * inf must not reach the accumulators where the last row's own weight does not.  (Widened: zeros.)
    const int tail_j = !U8 && te * TOK > kv_len ? cnt - 1 : -1;
    auto clear_tail = [&](uint8_t* slot) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
            if ((te - 1) * TOK + my_row + 4 * i >= kv_len) *reinterpret_cast<u4v*>(slot + wv * 2048 + i * 1024 + lane * 16) = u4v{0u, 0u, 0u, 0u};
    };
    __syncthreads();  // first_row
    const Rows r0 = row_of(0), r1 = row_of(1);
    Rows r2 = row_of(2), r3 = row_of(3);  // of the blocks j + 2 and j + 3
    copy_h(0, h0);
    copy_k(r0, k0);
    copy_v(r0, v0);
    copy_h(1, h1);
    copy_k(r1, k1);
    copy_v(r1, v1);
    copy_k(r2, k2);
    wait_vmem<0>();  // (the query loads as well)
#define PA_DENSE_STEP(KC, VC, HC, VP, KN, VN, HN)                                    \
    {                                                                                \
        lds_barrier();                                                               \
        copy_h(j + 2, HN);                                                           \
        copy_k(r3, KN);                                                              \
        copy_v(r2, VN);                                                              \
        if (j < cnt) qk(KC);                                                         \
        if (j > 0) pv(VP);                                                           \
        if (j == cnt) break;                                                         \
        wait_vmem<COPIES>();                                                         \
        if (j == tail_j) clear_tail(VC);                                             \
        r2 = r3;                                                                     \
        r3 = row_of(j + 4);                                                          \
        softmax(j, HC);                                                              \
        ++j;                                                                         \
    }
    for (int j = 0;;) {
        PA_DENSE_STEP(k0, v0, h0, v3, k3, v2, h2)
        PA_DENSE_STEP(k1, v1, h1, v0, k0, v3, h3)
        PA_DENSE_STEP(k2, v2, h2, v1, k1, v0, h0)
        PA_DENSE_STEP(k3, v3, h3, v2, k2, v1, h1)
    }
#undef PA_DENSE_STEP
    wait_vmem<0>();  // the clamped copies of the last steps still target this workgroup's LDS

    // ---- write the rows -----------------------------------------------------------------------------------------
    const bool final_out = item.nsplit == 1;
#pragma unroll
    for (int gi = 0; gi < NG; ++gi) {
        const float l = xor_sum_g(l_part[gi]);
        if (U8) {
            const float z = xor_sum_g(zsum[gi]);
#pragma unroll
            for (int r = 0; r < RT; ++r) acc[gi][r] = acc[gi][r] - z;
        }
        const float m_run = neg_m[gi] == NO_MAX ? -INFINITY : -neg_m[gi];
        if (row_pos[gi] < 0) continue;
        // register i of tile r on lane (n, g) holds channel 16 r + 4 g + i of row n
        if (final_out) {
            const float inv = l > 0.0f ? 1.0f / l : 0.0f;
            uint16_t* o = a.out + (long)row_id[gi] * HD;
#pragma unroll
            for (int r = 0; r < RT; ++r)
                *reinterpret_cast<uint2*>(o + 16 * r + 4 * g) = make_uint2(pack2<QDT>(acc[gi][r][0] * inv, acc[gi][r][1] * inv),
                                                                           pack2<QDT>(acc[gi][r][2] * inv, acc[gi][r][3] * inv));
            if (g == 0) {  // natural-log maximum and denominator for the score kernels
                a.final_ml[2 * (long)row_id[gi]] = m_run * LN2;
                a.final_ml[2 * (long)row_id[gi] + 1] = l;
            }
        } else {
            const long slot = (long)row_id[gi] * a.max_split + item.split;
            float* o = a.part_acc + slot * HD;
#pragma unroll
            for (int r = 0; r < RT; ++r) *reinterpret_cast<f4*>(o + 16 * r + 4 * g) = acc[gi][r];
            if (g == 0) {
                a.part_ml[2 * slot] = m_run;
                a.part_ml[2 * slot + 1] = l;
            }
        }
    }
}

// u8 rows -> rows of f16 integers, code - c with c the integer nearest the row's zero-point (|code - c| <= 255: exact, and
// normal numbers), and per token K scale x logit scale | -(zero-point - c) of K x that | V scale | zero-point - c of V.  One
// workgroup per (32-token block, kv head, listed sequence): eight threads to a row, sixteen codes of K and of V each.  Rows
// beyond the sequence's tokens are zeros.
__global__ __launch_bounds__(256) void pa_widen_kernel(WidenArgs a) {
    const WidenSeq ws = a.seqs[blockIdx.z];
    const int tile = ws.lo + blockIdx.x;
    if (tile >= ws.hi) return;
    const int hkv = blockIdx.y, row = threadIdx.x >> 3, part = threadIdx.x & 7;
    const int pos = tile * TOK + row, kv_len = a.st.past_lens[ws.b] + a.st.subsequence_begins[ws.b + 1] - a.st.subsequence_begins[ws.b];
    const bool live = pos < kv_len;
    const int at = min(pos, kv_len - 1), shift = 31 - __builtin_clz(a.sh.bs);
    const int id = a.block_indices[a.st.block_indices_begins[ws.b] + (at >> shift)];
    const long src = (((long)id * a.sh.Hkv + hkv) * a.sh.bs + (at & (a.sh.bs - 1))) * (HD + 8);
    const long dst = ((long)(ws.tile0 + tile) * a.sh.Hkv + hkv);
    float sc[2], z[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        const uint8_t* r = (t ? a.value_cache : a.key_cache) + src;
        const float2 h = *reinterpret_cast<const float2*>(r);
        const uint2 w0 = *reinterpret_cast<const uint2*>(r + 8 + 16 * part), w1 = *reinterpret_cast<const uint2*>(r + 16 + 16 * part);
        typedef _Float16 h2 __attribute__((ext_vector_type(2)));
        const float c = rintf(fminf(fmaxf(h.y, 0.0f), 255.0f));
        const _Float16 neg = (_Float16)(-1024.0f - c);
        const uint32_t w[4] = {w0.x, w0.y, w1.x, w1.y};
        u4v o[2];
#pragma unroll
        for (int i = 0; i < 4; ++i) {  // (0x64cc is 1024 + cc in f16)
            const h2 p = __builtin_bit_cast(h2, __builtin_amdgcn_perm(0x64646464u, w[i], 0x04010400u)) + h2{neg, neg};
            const h2 q = __builtin_bit_cast(h2, __builtin_amdgcn_perm(0x64646464u, w[i], 0x04030402u)) + h2{neg, neg};
            o[i >> 1][2 * (i & 1)] = live ? __builtin_bit_cast(uint32_t, p) : 0u;
            o[i >> 1][2 * (i & 1) + 1] = live ? __builtin_bit_cast(uint32_t, q) : 0u;
        }
        u4v* out = reinterpret_cast<u4v*>((t ? a.wide_v : a.wide_k) + dst * TILEB + row * ROWB + 32 * part);
        out[0] = o[0];
        out[1] = o[1];
        sc[t] = live ? h.x : 0.0f;
        z[t] = live ? h.y - c : 0.0f;
    }
    if (part == 0) {
        float* hdr = a.wide_hdr + dst * (HDRB / 4) + row;
        const float s = sc[0] * (a.st.scale * LOG2E);
        hdr[0] = s;
        hdr[TOK] = -z[0] * s;
        hdr[2 * TOK] = sc[1];
        hdr[3 * TOK] = z[1];
    }
}
}  // namespace

hipError_t launch_widen(hipStream_t s, const WidenArgs& a) {
    hipLaunchKernelGGL(pa_widen_kernel, dim3((unsigned)a.max_tiles, (unsigned)a.sh.Hkv, (unsigned)a.n_seqs), dim3(256), 0, s, a);
    return hipGetLastError();
}

hipError_t launch_prefill_dense(hipStream_t s, const PrefillArgs& a, int q_dtype, bool widened) {
    if (a.sh.D != HD || a.G > PREFILL_ROWS) return hipErrorInvalidValue;
    const dim3 grid((unsigned)a.n_items * a.sh.Hkv);
    if (widened) {
        if (q_dtype == DT_F16) hipLaunchKernelGGL((pa_prefill_dense_kernel<DT_F16, DT_F16, true>), grid, dim3(64 * NW), 0, s, a);
        else hipLaunchKernelGGL((pa_prefill_dense_kernel<DT_F16, DT_BF16, true>), grid, dim3(64 * NW), 0, s, a);
    } else if (q_dtype == DT_F16) {
        hipLaunchKernelGGL((pa_prefill_dense_kernel<DT_F16, DT_F16, false>), grid, dim3(64 * NW), 0, s, a);
    } else {
        hipLaunchKernelGGL((pa_prefill_dense_kernel<DT_BF16, DT_BF16, false>), grid, dim3(64 * NW), 0, s, a);
    }
    return hipGetLastError();
}

}  // namespace pa
