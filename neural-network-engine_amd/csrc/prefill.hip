// FlashAttention forward for gfx950: f32 on the bf16 matrix cores.
//
// Algorithm: the tiled online softmax of the reference's
// flash_attention_forward (src/nn/flash_attention.rs:91-195) -- per query row a
// running max m and sum l, P = exp(S - m), O = alpha*O + P V, O /= l at the end
// with rows that saw no key left at zero (:186-194), fully masked key tiles
// skipped (:101-104) -- generalised to grouped-query heads (KV head hq / G) and
// a causal offset.
//
// MI355X mapping (head dims up to 128; 129-512 dims: prefill_wide_kernel).
// Every f32 operand is the exact sum of three bf16 parts and every product the
// six largest products of parts (nne_common.hpp), on v_mfma_f32_32x32x16_bf16.
// One wave owns 32 query rows and computes the score tile transposed,
// S^T = K Q^T:
//   A = K tile  (lane l supplies key l%32, dims 16t + 8*(l/32) + 0..7 of step t)
//   B = Q^T     (lane l supplies query row l%32; held in registers, pre-scaled
//                by scale*log2(e) so the softmax is a bare exp2)
// The accumulator layout of S^T puts query row l%32 in lane l and keys
// 8*(r/4) + 4*(l/32) + r%4 in register r, so
//   * the row max / row sum are 16 in-lane ops plus one lane-pair exchange
//     (v_permlane32_swap),
//   * the parts of P^T registers 8s .. 8s + 7 are already the B operand of step
//     s of O^T = V^T P^T (V's keys are laid out to match), so P never leaves
//     registers,
//   * every O^T accumulator of a lane belongs to that lane's query row, so the
//     online-softmax rescale is a lane-local multiply -- done lazily, only
//     when a row max grows by more than 2^8.
// K and V tiles (32 keys) are split into their parts by the threads that load
// them, once per workgroup, and left in LDS in operand order: 6 bytes a value.
// One buffer each for K and V: a tile's K is replaced while its softmax and
// P V run, its V while the next S^T runs, each from registers loaded a phase
// before, with a barrier between the phases; at D = 128 two workgroups (49 KB
// of tiles each) share a CU and fill each other's waits.  The G query heads
// that share a KV head run as waves of one workgroup and read the same staged
// tiles.  Workgroups are numbered so that each XCD works on a contiguous range
// of KV heads (its own L2) and, within a head, the longest causal row blocks
// start first.
//
// What bounds it: the matrix cores, and the power they draw.  A tile takes a
// wave 96 MFMAs of 32 cycles at D = 128 beside about 340 vector instructions
// (softmax, the parts of P, K and V); with random operands a stream of nothing
// but these MFMAs settles at 1777 TFLOP/s, 296 TFLOP/s of f32 products.
// Measured against the f32 MFMAs (v_mfma_f32_32x32x2, 157 TFLOP/s at most):
// B = 4, Hq = 32, Hkv = 8, T = 2048, d = 128 causal 1075 -> 697-717 us, B =
// 1, H = 16, T = 16384, d = 64 causal 4346 -> 2810-2970 us, B = 8, H = 20, T =
// 1500, d = 64 777 -> 484 us, with 0.4 to 0.9 of the error against 64 bits.
//
// Problems with fewer work items than CUs instead cut each item's key tiles
// into chunks, one workgroup per (item, chunk); the last chunk of an item to
// finish folds the partial (max, sum, O) records in chunk order (the same
// combine as the online softmax, so the result is independent of arrival
// order) and writes O.
#include <atomic>
#include <utility>
#include <vector>

#include "nne_common.hpp"
#include "nne_launch.hpp"

namespace nne {

namespace {

// Last key index visible to any row of row block rb (or -1).
__device__ __forceinline__ int last_visible_key(const PrefillParams& p, int rb, bool causal) {
    if (!causal) return p.Tk - 1;
    int last_row = rb * 32 + 31;
    if (last_row > p.Tq - 1) last_row = p.Tq - 1;
    int lk = last_row + p.q_offset;
    return lk < p.Tk - 1 ? lk : p.Tk - 1;
}

// The j-th work item of the workgroup in slot q of XCD x (S slots per XCD):
// super-items x*per_xcd + q + k*S, k = 0, 1, ..., each one item (rank pr) or,
// with pairing, two (ranks pr and n_wg-1-pr).  Rank r is wgi = n_wg-1-r, so
// rank 0 holds the longest causal rows.  Returns 0 past the end, 2 for the
// missing partner of an odd middle rank, 1 with (head, wgi) otherwise.
__device__ __forceinline__ int item_at(const PrefillParams& p, int j, int x, int q, int S, int& head,
                                       int& wgi) {
    if (p.order_all) {
        const int heads = p.B * p.Hkv, i = 8 * q + x;
        if (j > 0 || i >= heads * p.n_wg) return 0;
        head = i % heads;
        wgi = p.n_wg - 1 - i / heads;
        return 1;
    }
    if (p.order_cu) {
        // Position pos in the XCD's items sorted longest first (rank-major over
        // its heads).  The hardware places workgroup q of an XCD on CU q % h
        // (h CUs, q < h first): with n <= 2h items the CUs that get a second
        // workgroup take a longer and a shorter item whose lengths add up to
        // about the same, and the CUs with one take the longest items.
        if (j > 0) return 0;
        const int h = p.order_cu, n = p.per_xcd;
        int pos = q;
        if (n <= 2 * h && n > h) {
            if (q >= h) pos = n - 1 - (q - h);
            else if (q >= n - h) pos = q - (n - h);
            else pos = (2 * h - n) + q;
        }
        head = x * p.order_hpx + pos % p.order_hpx;
        wgi = p.n_wg - 1 - pos / p.order_hpx;
        return 1;
    }
    const int k = p.pairing ? j >> 1 : j;
    const int s = x * p.per_xcd + q + k * S;
    int s_end = (x + 1) * p.per_xcd;
    if (s_end > p.n_super) s_end = p.n_super;
    if (s >= s_end) return 0;
    head = s / p.n_pairs;
    const int pr = s % p.n_pairs;
    int rank = pr;
    if (p.pairing && (j & 1)) {
        rank = p.n_wg - 1 - pr;
        if (rank == pr) return 2;
    }
    wgi = p.n_wg - 1 - rank;
    return 1;
}

// K/V tile of 32 keys x D dims, read by 4 or 8 waves and left in LDS as three
// bf16 planes each, in operand order (one 16-byte slot per lane):
//   K (A of S^T = K Q^T): plane p, 16-dim step t, lane half h, key r at slot
//     (p * D/16 + t) * 64 + h * 32 + (r ^ ((2t + h) & 15)), dims 16t + 8h .. + 7.
//     The XOR spreads the 16 slots that one key's dims are stored to over the
//     banks; a step's reads stay one contiguous 1 KB.
//   V (A of O^T = V^T P^T): plane p, 32-dim block b, 16-key step s, lane half
//     h, dim m at slot ((p * NB + b) * 2 + s) * 64 + h * 32 + m, keys
//     16s + 4h + 0..3 and 16s + 8 + 4h + 0..3 (the keys of lane half h in
//     registers 8s .. 8s + 7 of the S^T accumulator).
// Rows past T_k are zeros, or with scalar loads row T_k - 1 again (their
// weights are zero); dims past d read dim 0 (Q is zero there, and those output
// dims are not stored).
template <int D, bool VEC, int WAVES = 4>
struct SplitTile {
    static constexpr int NB = D / 32;
    static constexpr int K_PLANE = 32 * D * 2, V_PLANE = 32 * D * 2;   // bytes
    static constexpr int LPR = D / 4;                      // lanes per key row (4 dims each)
    static constexpr int NC = (LPR + 63) / 64;            // loads per key row
    static constexpr int RPI = LPR <= 64 ? 64 / LPR : 1;   // rows per load
    static constexpr int KR = 32 / WAVES;                  // key rows per wave
    static constexpr int NK = KR / RPI * NC;               // K loads per thread
    static constexpr int VD = D / (WAVES / 4);             // dims per wave of V
    static constexpr int NJ = (VD + 63) / 64;              // dims per lane of V
    static_assert(KR % RPI == 0 && LPR <= 64 * NC, "whole rows per load");
    float4 kr[NK];
    float vr[NJ][8];
    // VEC views (row strides in [0, kMaxTileStride)): byte offsets of this lane within a
    // tile and of each load's rows, so that a tile's loads need only its base.
    uint32_t k_lane[NC], k_step, v_lane[NJ], v_row0, v_st;

    // This lane's row among a load's and its first dim in load column j (a row
    // of 96 dims leaves the lanes past two rows to repeat the second).
    static __device__ __forceinline__ int row_of(int lane) { return min(lane / LPR, RPI - 1); }
    static __device__ __forceinline__ int col_of(int lane, int j) {
        return NC > 1 ? min((lane + 64 * j) * 4, D - 4) : lane < LPR * RPI ? (lane % LPR) * 4 : D - 4;
    }
    static __device__ __forceinline__ int dim_of(int wave, int lane, int j) {
        return (wave >> 2) * VD + lane + 64 * j;
    }

    __device__ __forceinline__ void init(const PrefillParams& p, int wave, int lane) {
        const uint32_t kst = (uint32_t)p.k.st * 4u, vst = (uint32_t)p.v.st * 4u;
#pragma unroll
        for (int j = 0; j < NC; ++j) {
            const int c = col_of(lane, j);
            k_lane[j] = (KR * wave + row_of(lane)) * kst + (c < p.d ? c : 0) * 4;
        }
        k_step = RPI * kst;
        v_row0 = (16 * ((wave >> 1) & 1) + 4 * (wave & 1)) * vst;
        v_st = vst;
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            const int dim = dim_of(wave, lane, j);
            v_lane[j] = (dim < p.d ? dim : 0) * 4;
        }
    }

    // Rows key0 .. key0 + 31 of a KV head, ending with the last key (rows past
    // it read as zeros without a memory access).
    // (Without a tile, ok false: an empty range.)
    static __device__ __forceinline__ __amdgpu_buffer_rsrc_t tile_range(const float* base, int64_t st,
                                                                        int key0, int Tk, int d, bool ok) {
        const int rows = min(32, Tk - key0);
        return __builtin_amdgcn_make_buffer_rsrc(
            const_cast<float*>(base + key0 * st), 0,
            ok ? ((rows - 1) * (uint32_t)st + d) * 4u : 0u, 0x00020000);
    }

    __device__ __forceinline__ void load_k(const PrefillParams& p, const float* kb, int key0,
                                           int wave, int lane, bool ok) {
        if (VEC) {
            const auto range = tile_range(kb, p.k.st, key0, p.Tk, p.d, ok);
            if (ok && key0 + 32 <= p.Tk) {
#pragma unroll
                for (int i = 0; i < NK; ++i)
                    kr[i] = __builtin_bit_cast(
                        float4, __builtin_amdgcn_raw_buffer_load_b128(range, k_lane[i % NC], i / NC * k_step, 0));
            } else {
                // (Whole offsets in the lanes: the check of the tail's rows takes in no other.)
#pragma unroll
                for (int i = 0; i < NK; ++i)
                    kr[i] = __builtin_bit_cast(
                        float4, __builtin_amdgcn_raw_buffer_load_b128(range, k_lane[i % NC] + i / NC * k_step, 0, 0));
            }
        } else if (ok) {
#pragma unroll
            for (int i = 0; i < NK; ++i) {
                int key = key0 + KR * wave + row_of(lane) + RPI * (i / NC);
                if (key > p.Tk - 1) key = p.Tk - 1;
                const float* a = kb + key * p.k.st;
                const int c = col_of(lane, i % NC);
                float t[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) t[j] = a[(c + j < p.d ? c + j : 0) * p.k.sd];
                kr[i] = make_float4(t[0], t[1], t[2], t[3]);
            }
        }
    }

    // The parts of one load (4 dims of a key) computed and stored, for the
    // caller to place between MFMAs; store_k does all NK.
    __device__ __forceinline__ void part_k(int i, char* ks, int wave, int lane) const {
        const int c4 = col_of(lane, i % NC) >> 2, c8 = c4 >> 1;   // 8-dim chunk 2t + h
        const int r = KR * wave + row_of(lane) + RPI * (i / NC);
        uint2 h, m, l;
        split3(kr[i].x, kr[i].y, h.x, m.x, l.x);
        split3(kr[i].z, kr[i].w, h.y, m.y, l.y);
        char* a = ks + c8 * 512 + (c4 & 1) * 8 + ((r ^ (c8 & 15)) << 4);
        *reinterpret_cast<uint2*>(a) = h;
        *reinterpret_cast<uint2*>(a + K_PLANE) = m;
        *reinterpret_cast<uint2*>(a + 2 * K_PLANE) = l;
    }
    __device__ __forceinline__ void store_k(char* ks, int wave, int lane) const {
#pragma unroll
        for (int i = 0; i < NK; ++i) part_k(i, ks, wave, lane);
    }

    // Wave w reads the 8 keys of (step s, lane half h) = (w / 2 % 2, w % 2); with
    // 8 waves, waves 4-7 the second half of the dims.
    __device__ __forceinline__ void load_v(const PrefillParams& p, const float* vb, int key0,
                                           int wave, int lane, bool ok) {
        if (VEC) {
            const auto range = tile_range(vb, p.v.st, key0, p.Tk, p.d, ok);
            if (ok && key0 + 32 <= p.Tk) {
#pragma unroll
                for (int i = 0; i < 8; ++i)
#pragma unroll
                    for (int j = 0; j < NJ; ++j)
                        vr[j][i] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(
                            range, v_lane[j], v_row0 + (8 * (i >> 2) + (i & 3)) * v_st, 0));
            } else {
#pragma unroll
                for (int i = 0; i < 8; ++i)
#pragma unroll
                    for (int j = 0; j < NJ; ++j)
                        vr[j][i] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(
                            range, v_lane[j] + v_row0 + (8 * (i >> 2) + (i & 3)) * v_st, 0, 0));
            }
        } else if (ok) {
            const int k0 = key0 + 16 * ((wave >> 1) & 1) + 4 * (wave & 1);
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                int key = k0 + 8 * (i >> 2) + (i & 3);
                if (key > p.Tk - 1) key = p.Tk - 1;
                const float* a = vb + key * p.v.st;
#pragma unroll
                for (int j = 0; j < NJ; ++j) {
                    const int dim = dim_of(wave, lane, j);
                    vr[j][i] = a[(dim < p.d ? dim : 0) * p.v.sd];
                }
            }
        }
    }

    // Likewise two keys of a dim; every fourth step stores the dim's 8 keys.
    uint32_t vp[3][4];
    __device__ __forceinline__ void part_v(int i, char* vs, int wave, int lane) {
        const int j = i >> 2, dim = dim_of(wave, lane, j);
        split3(vr[j][2 * (i & 3)] * kPartUp, vr[j][2 * (i & 3) + 1] * kPartUp, vp[0][i & 3], vp[1][i & 3],
               vp[2][i & 3]);
        if ((i & 3) != 3 || (64 * (j + 1) > VD && lane + 64 * j >= VD)) return;
        char* a = vs + (((dim >> 5) * 2 + ((wave >> 1) & 1)) * 64 + (wave & 1) * 32 + (dim & 31)) * 16;
#pragma unroll
        for (int u = 0; u < 3; ++u)
            *reinterpret_cast<uint4*>(a + u * V_PLANE) = make_uint4(vp[u][0], vp[u][1], vp[u][2], vp[u][3]);
    }
    __device__ __forceinline__ void store_v(char* vs, int wave, int lane) {
#pragma unroll
        for (int i = 0; i < 4 * NJ; ++i) part_v(i, vs, wave, lane);
    }
};

template <int NB>
__device__ __forceinline__ bool finite(const floatx16 (&o)[NB]) {
    uint32_t most = 0;
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r) most = max(most, __float_as_uint(o[b][r]) & 0x7fffffffu);
    return most < 0x7f800000u;
}

// One 32-row unit (its output dims dim0 .. dim0 + 32 NB - 1) over key tiles
// [t0, t1) in plain f32 MFMAs on operands read from global memory: the arithmetic
// for inputs outside the range of the parts (infinities, NaN, magnitudes near the
// top of f32's; scaled queries beyond 2^90 or below 2^-110).  Everything it needs
// is derived here from a few opaque scalars, so that nothing of it is computed
// ahead of, or kept in registers across, the main loop.
//
// What bounds it: its loads, 32 dims of K and Q or 4 keys of V at a time before 16
// MFMAs or more.  With one NaN in every head's V, so that every unit comes here
// after the bf16 products (us; without it; one dim pair and one key at a time;
// all f32 from the start on K/V tiles in LDS): d = 64, B = 4, H = 20, T = 300 62 (26,
// 108, 29); d = 128 108 (41, 216, 53); d = 256, H = 140, T = 97 95 (36, 213, 47);
// d = 512 253 (81, 554, 82).
template <int D, int NB, bool CAUSAL, bool VEC>
__device__ __forceinline__ void unit_f32(const PrefillParams& p, int head, int unit, int t0, int t1,
                                         int dim0, floatx16 (&o)[NB], float& m_run, float& l_run) {
    constexpr int NL = D == 32 ? 2 : 4;   // loads of K and Q at a time (32 dims: four workgroups per CU)
    int tid = threadIdx.x;
    float zero = 0.f;
    asm volatile("" : "+v"(tid), "+v"(zero), "+s"(head), "+s"(unit), "+s"(t0), "+s"(t1),
                 "+s"(dim0));
    const int l32 = tid & 31, half = (tid >> 5) & 1;
    const int bi = head / p.Hkv, kvh = head % p.Hkv;
    const int qrow = unit / p.G * 32 + l32;
    const bool rok = qrow < p.Tq;
    const float* qp = p.q.p + bi * p.q.sb + (kvh * p.G + unit % p.G) * p.q.sh + (int64_t)qrow * p.q.st;
    const float* kb = p.k.p + bi * p.k.sb + kvh * p.k.sh;
    const float* vb = p.v.p + bi * p.v.sb + kvh * p.v.sh;
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[b][r] = zero;
    m_run = kNegInf;
    l_run = zero;
    // Dims c .. c + 3 of a row (zeros past the last dim or row).
    const auto load4 = [&](const float* row, int64_t sd, int c, bool ok) {
        vf4 x = {0.f, 0.f, 0.f, 0.f};
        if (VEC) {
            if (ok && c < p.d) x = *reinterpret_cast<const vf4*>(row + c);
        } else {
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (ok && c + j < p.d) x[j] = row[(c + j) * sd];
        }
        return x;
    };
#pragma nounroll
    for (int kt = t0; kt < t1; ++kt) {
        const int key0 = kt * 32;
        const bool kok = key0 + l32 < p.Tk;
        const float* kp = kb + (int64_t)(kok ? key0 + l32 : 0) * p.k.st;
        int c0 = 4 * half;
        asm volatile("" : "+v"(c0));   // Q is read again each tile, not held across them
        // Two sums per score: half the roundings in each.
        floatx16 s, s2;
#pragma unroll
        for (int r = 0; r < 16; ++r) s[r] = s2[r] = zero;
#pragma nounroll
        for (int t = 0; t < D; t += 8 * NL) {
            vf4 kx[NL], qx[NL];
#pragma unroll
            for (int i = 0; i < NL; ++i) kx[i] = load4(kp, p.k.sd, t + 8 * i + c0, kok);
#pragma unroll
            for (int i = 0; i < NL; ++i) qx[i] = load4(qp, p.q.sd, t + 8 * i + c0, rok);
#pragma unroll
            for (int i = 0; i < NL; ++i)
#pragma unroll
                for (int j = 0; j < 4; j += 2) {
                    s = __builtin_amdgcn_mfma_f32_32x32x2f32(kx[i][j], qx[i][j] * p.qscale, s, 0, 0, 0);
                    s2 = __builtin_amdgcn_mfma_f32_32x32x2f32(kx[i][j + 1], qx[i][j + 1] * p.qscale, s2, 0, 0, 0);
                }
        }
        float mt = kNegInf;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int key = key0 + 8 * (r >> 2) + 4 * half + (r & 3);
            const bool vis = key < p.Tk && (!CAUSAL || key <= qrow + p.q_offset);
            s[r] = vis ? s[r] + s2[r] : kNegInf;
            mt = fmaxf(mt, s[r]);
        }
        const float m_new = fmaxf(m_run, pair_max(mt));
        const float m_use = m_new == kNegInf ? 0.f : m_new;
        const float alpha = fast_exp2(m_run - m_use);
        l_run *= alpha;
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int r = 0; r < 16; ++r) o[b][r] *= alpha;
        m_run = m_new;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            // Four keys' V in registers at a time.
            float vx[4][NB];
            int key = key0 + 8 * g + 4 * half;
            asm volatile("" : "+v"(key));
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const bool ok = key + j < p.Tk;
                const float* vp = vb + (int64_t)(ok ? key + j : 0) * p.v.st;
#pragma unroll
                for (int b = 0; b < NB; ++b) {
                    const int dim = dim0 + 32 * b + l32;
                    vx[j][b] = ok && dim < p.d ? vp[dim * p.v.sd] : 0.f;
                }
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float pr = fast_exp2(s[4 * g + j] - m_use);
                l_run += pr;
#pragma unroll
                for (int b = 0; b < NB; ++b)
                    o[b] = __builtin_amdgcn_mfma_f32_32x32x2f32(vx[j][b], pr, o[b], 0, 0, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }
}

// Two workgroups per CU, three up to 64 dims for the persistent schedule.  At
// d = 128 the scalar-load variant (views that are not 16-byte vectors) takes the
// whole register file instead of spilling.
template <int D, bool CAUSAL, bool VEC, bool SPLIT>
__global__ __launch_bounds__(256, D >= 128 && !VEC ? 1 : D <= 64 && !SPLIT ? 3 : 2) void prefill_mfma_kernel(const PrefillParams p) {
    using Tile = SplitTile<D, VEC>;
    constexpr int NB = D / 32;         // 32-wide output column blocks
    constexpr int NT = D / 16;         // 16-dim steps of S^T
    constexpr int KP = Tile::K_PLANE, VP = Tile::V_PLANE;
    // At D = 128 the low parts of Q's last steps stay in LDS (16 registers that
    // the two-wave budget of 256 does not hold).
    constexpr int NQL = D == 128 && VEC ? 4 : 0;
    __shared__ __attribute__((aligned(16))) char lds[3 * (KP + VP) + NQL * 4096];
    char* const Ks = lds;
    char* const Vs = lds + 3 * KP;
    char* const Qs = Vs + 3 * VP;

    // Every argument's cache line in one round trip (left to the compiler, the
    // first uses and the search below pay one each).
    warm_kernargs<0, SPLIT ? sizeof(PrefillParams) : offsetof(PrefillParams, part_prefix)>();

    // ---- persistent workgroup: slot q of XCD x -------------------------------
    // Hardware dispatches consecutive workgroup ids round-robin over the 8
    // XCDs, so x = id & 7; each XCD owns a contiguous range of super-items
    // (whole KV heads, its own L2).  The workgroup runs its items one after the
    // other: no dispatch gaps, and the static schedule is balanced.
    const int x = blockIdx.x & 7, q = blockIdx.x >> 3, S = gridDim.x >> 3;

#pragma nounroll
    for (int j = 0;; ++j) {
    int head = 0, wgi = 0, chunk = 0, pair = 0;
    int n_parts = 1;
    if constexpr (SPLIT) {
        // Key split, one step only.  The (item, chunk) pairs are numbered
        // contiguously per head; XCD x (= workgroup id % 8, the hardware's
        // dealing order) takes the x-th eighth of that list, so the chunks of
        // an item share one L2 (they all read the item's Q).
        if (j > 0) break;
        const int per_head = p.part_prefix[p.n_wg];
        const int pairs = p.B * p.Hkv * per_head;
        const int ppx = (pairs + 7) >> 3;
        pair = (blockIdx.x & 7) * ppx + (blockIdx.x >> 3);
        if (pair >= pairs) break;
        head = pair / per_head;
        const int r = pair % per_head;
        int lo = 0, hi = p.n_wg - 1;     // last item with part_prefix <= r
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (p.part_prefix[mid] <= r) lo = mid; else hi = mid - 1;
        }
        wgi = lo;
        chunk = r - p.part_prefix[lo];
        n_parts = p.part_prefix[lo + 1] - p.part_prefix[lo];
    } else {
        const int st = item_at(p, j, x, q, S, head, wgi);
        if (st == 0) break;
        if (st == 2) continue;
    }
    // Lane-derived addressing is recomputed for every item rather than held
    // live across the whole persistent loop.
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, half = lane >> 5;
    const int bi = head / p.Hkv, kvh = head % p.Hkv;

    const int unit = wgi * 4 + wave;
    const bool active = unit < p.n_units;
    const int rb = active ? unit / p.G : 0;
    const int g = active ? unit % p.G : 0;
    const int hq = kvh * p.G + g;
    const int row0 = rb * 32;
    const int qrow = row0 + l32;

    // ---- key-tile range ------------------------------------------------------
    const int n_kt = (p.Tk + 31) >> 5;
    int last_unit = wgi * 4 + 3;
    if (last_unit > p.n_units - 1) last_unit = p.n_units - 1;
    const int wg_last_key = last_visible_key(p, last_unit / p.G, CAUSAL);
    int n_tiles = wg_last_key < 0 ? 0 : (wg_last_key >> 5) + 1;
    if (n_tiles > n_kt) n_tiles = n_kt;
    const int wave_last_key = last_visible_key(p, rb, CAUSAL);
    const int wave_tiles = active ? (wave_last_key < 0 ? 0 : (wave_last_key >> 5) + 1) : 0;

    // Key tiles [t0, t1) of this workgroup: all of them, or one chunk (an
    // empty chunk still leaves its record).
    int t0 = 0, t1 = n_tiles;
    if constexpr (SPLIT) {
        t0 = min(n_tiles, chunk * p.chunk_tiles);
        t1 = min(n_tiles, t0 + p.chunk_tiles);
    }

    const float* kb = p.k.p + bi * p.k.sb + kvh * p.k.sh;
    const float* vb = p.v.p + bi * p.v.sb + kvh * p.v.sh;

    // The second item of a causal pair walks its key tiles backwards.  The
    // workgroups of an XCD then stand at only two key positions at any time
    // -- t on their first (long) items, total - t on their second (short)
    // ones, whatever their ranks -- so the head's K/V tiles they read stay in
    // the XCD's L2.  Walked forwards, every second item restarts at key 0 at
    // its own time and the walks spread over the whole head: B = 1, H = 16, T =
    // 16384, d = 64 read 284 MB from HBM, 249 MB backwards on the f32 MFMAs (201 MB
    // algorithmic), same time; 350 MB now.
    const bool rev = !SPLIT && p.pairing && (j & 1);
    const int kstep = rev ? -1 : 1;
    const int kfirst = rev ? t1 - 1 : t0;
    const int n_it = t1 - t0;
    Tile ld;
    ld.init(p, wave, lane);
    // The first tile's loads go before Q's, so that the two latencies overlap.
    if (n_it > 0) {
        ld.load_k(p, kb, kfirst * 32, wave, lane, true);
        ld.load_v(p, vb, kfirst * 32, wave, lane, true);
    }

    // ---- Q^T: three bf16 parts of Q[qrow][16t + 8*half + 0..7] * scale*log2(e)
    short8 qf[2][NT], ql[NT - NQL];
    char* const qls = Qs + (wave * NQL * 64 + lane) * 16;
    const float* qp = p.q.p + bi * p.q.sb + hq * p.q.sh + (int64_t)qrow * p.q.st;
    const bool rok = active && qrow < p.Tq;
    uint32_t q_code = 0;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        const int c = 16 * t + 8 * half;
        float x[8];
#pragma unroll
        for (int j = 0; j < 8; j += 4) {
            if (VEC) {
                const float4 t4 = (rok && c + j < p.d) ? *reinterpret_cast<const float4*>(qp + c + j)
                                                       : make_float4(0.f, 0.f, 0.f, 0.f);
                x[j] = t4.x; x[j + 1] = t4.y; x[j + 2] = t4.z; x[j + 3] = t4.w;
            } else {
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    x[j + u] = (rok && c + j + u < p.d) ? qp[(c + j + u) * p.q.sd] : 0.f;
            }
        }
        uint4 h, m, l;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            x[j] *= p.qscale;
            q_code = max(q_code, range_code(x[j]));
        }
        split3(x[0], x[1], h.x, m.x, l.x);
        split3(x[2], x[3], h.y, m.y, l.y);
        split3(x[4], x[5], h.z, m.z, l.z);
        split3(x[6], x[7], h.w, m.w, l.w);
        qf[0][t] = __builtin_bit_cast(short8, h);
        qf[1][t] = __builtin_bit_cast(short8, m);
        if (t < NT - NQL) ql[t < NT - NQL ? t : 0] = __builtin_bit_cast(short8, l);
        else *reinterpret_cast<uint4*>(qls + (t - (NT - NQL)) * 1024) = l;
    }
    asm volatile("" : "+v"(q_code));   // computed here, not from every x after the loop

    floatx16 o[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[b][r] = 0.f;
    float m_run = kNegInf, l_run = 0.f;

    if (n_it > 0) {
        ld.store_k(Ks, wave, lane);
        ld.store_v(Vs, wave, lane);
    }
    __syncthreads();

    for (int it = 0; it < n_it; ++it) {
        const int kt = kfirst + kstep * it;
        const bool has_next = it + 1 < n_it;
        const bool mine = kt < wave_tiles;
        ld.load_k(p, kb, (kt + kstep) * 32, wave, lane, has_next);
        floatx16 s;
        const float m_use = (m_run == kNegInf) ? 0.f : m_run;
        if (mine) {
            // S^T = K Q^T  (32 keys x 32 rows), log2 domain: first every small
            // product, then the products of the high parts, so that only D/16 sums
            // are rounded at the size of the score.  (Sums that start at -m are all
            // rounded at m's.  Error against 64 bits at d = 128 with 200 in every
            // score, spread over the dims: 3.7e-6, from -m 2.3e-5, on the f32 MFMAs
            // 1.8e-5; N(0, 1) operands 2.3e-7, 4.7e-7, 4.9e-7.  It costs 16
            // subtractions in the softmax: d = 64, T = 16384 0.5 %.)
#pragma unroll
            for (int r = 0; r < 16; ++r) s[r] = 0.f;
            const int kbase = half * 512 + ((l32 ^ half) << 4);
            // Raised issue priority while this wave feeds the MFMA pipe, so the
            // two waves sharing a SIMD alternate MFMA and softmax phases.
            __builtin_amdgcn_s_setprio(1);
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                const char* a = Ks + t * 1024 + (kbase ^ ((2 * t & 15) << 4));
                const short8 kh = *reinterpret_cast<const short8*>(a);
                const short8 km = *reinterpret_cast<const short8*>(a + KP);
                const short8 kl = *reinterpret_cast<const short8*>(a + 2 * KP);
                s = mfma_bf16(kl, qf[0][t], s);
                s = mfma_bf16(kh, t < NT - NQL ? ql[t < NT - NQL ? t : 0]
                                               : *reinterpret_cast<const short8*>(
                                                     qls + (t - (NT - NQL)) * 1024), s);
                s = mfma_bf16(km, qf[1][t], s);
                s = mfma_bf16(km, qf[0][t], s);
                s = mfma_bf16(kh, qf[1][t], s);
            }
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                const char* a = Ks + t * 1024 + (kbase ^ ((2 * t & 15) << 4));
                s = mfma_bf16(*reinterpret_cast<const short8*>(a), qf[0][t], s);
            }
            // Schedule: the operands of a step are read one step ahead.
            __builtin_amdgcn_sched_group_barrier(0x100, 3, 0);
#pragma unroll
            for (int t = 0; t < NT - 1; ++t) {
                if (t + 1 < NT - NQL) __builtin_amdgcn_sched_group_barrier(0x100, 3, 0);
                else __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
                __builtin_amdgcn_sched_group_barrier(0x008, 5, 0);
            }
            __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, 5, 0);
#pragma unroll
            for (int t = 0; t < NT - 2; ++t) {
                __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            }
            __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
            __builtin_amdgcn_s_setprio(0);
        }
        __syncthreads();   // every wave has read K; V is visible
        if (has_next) ld.store_k(Ks, wave, lane);
        ld.load_v(p, vb, (kt + kstep) * 32, wave, lane, has_next);
        if (mine) {
            // Mask keys past T_k and (causal) keys after row + q_offset.
            const int key0 = kt * 32;
            const bool need_mask = (key0 + 32 > p.Tk) || (CAUSAL && key0 + 31 > row0 + p.q_offset);
            if (need_mask) {
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int key = key0 + 8 * (r >> 2) + 4 * half + (r & 3);
                    const bool vis = key < p.Tk && (!CAUSAL || key <= qrow + p.q_offset);
                    s[r] = vis ? s[r] : kNegInf;
                }
            }

            // Online softmax for this lane's row (keys split over the lane pair).
            // m_run is the reference max the exponentials use.  It is raised,
            // and O and l rescaled, only when some row's tile max exceeds it by
            // more than 8 (log2 units): P values stay <= 2^8, the ratio O/l is
            // unchanged, and most tiles skip the 4*NB*4 multiplies.
#pragma unroll
            for (int r = 0; r < 16; ++r) s[r] -= m_use;
            float mt = s[0];
#pragma unroll
            for (int r = 1; r < 16; ++r) mt = fmaxf(mt, s[r]);
            mt = pair_max(mt);
            if (__builtin_amdgcn_ballot_w64(mt > (m_run == kNegInf ? kNegInf : 8.f)) != 0) {
                const float m_new = fmaxf(m_run, mt + m_use);
                const float n_use = (m_new == kNegInf) ? 0.f : m_new;
                const float alpha = fast_exp2(m_run - n_use);
                l_run *= alpha;
#pragma unroll
                for (int b = 0; b < NB; ++b)
#pragma unroll
                    for (int r = 0; r < 16; ++r) o[b][r] *= alpha;
#pragma unroll
                for (int r = 0; r < 16; ++r) s[r] -= n_use - m_use;
                m_run = m_new;
            }
            float ls = 0.f;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                s[r] = fast_exp2(s[r]);
                ls += s[r];
            }
            l_run += ls;

            // O^T += V^T P^T ; step st takes the keys of registers 8st .. 8st+7.
            __builtin_amdgcn_s_setprio(1);
#pragma unroll
            for (int st = 0; st < 2; ++st) {
                uint4 h, m, l;
                split3(s[8 * st + 0] * kPartUp, s[8 * st + 1] * kPartUp, h.x, m.x, l.x);
                split3(s[8 * st + 2] * kPartUp, s[8 * st + 3] * kPartUp, h.y, m.y, l.y);
                split3(s[8 * st + 4] * kPartUp, s[8 * st + 5] * kPartUp, h.z, m.z, l.z);
                split3(s[8 * st + 6] * kPartUp, s[8 * st + 7] * kPartUp, h.w, m.w, l.w);
                const short8 ph = __builtin_bit_cast(short8, h), pm = __builtin_bit_cast(short8, m),
                             pl = __builtin_bit_cast(short8, l);
#pragma unroll
                for (int b = 0; b < NB; ++b) {
                    const char* a = Vs + ((b * 2 + st) * 64 + lane) * 16;
                    const short8 vh = *reinterpret_cast<const short8*>(a);
                    const short8 vm = *reinterpret_cast<const short8*>(a + VP);
                    const short8 vl = *reinterpret_cast<const short8*>(a + 2 * VP);
                    o[b] = mfma_bf16(vl, ph, o[b]);
                    o[b] = mfma_bf16(vh, pl, o[b]);
                    o[b] = mfma_bf16(vm, pm, o[b]);
                    o[b] = mfma_bf16(vm, ph, o[b]);
                    o[b] = mfma_bf16(vh, pm, o[b]);
                    o[b] = mfma_bf16(vh, ph, o[b]);
                }
            }
            __builtin_amdgcn_sched_group_barrier(0x100, 3, 0);
#pragma unroll
            for (int i = 0; i < 2 * NB - 1; ++i) {
                __builtin_amdgcn_sched_group_barrier(0x100, 3, 0);
                __builtin_amdgcn_sched_group_barrier(0x008, 6, 0);
            }
            __builtin_amdgcn_sched_group_barrier(0x008, 6, 0);
            __builtin_amdgcn_s_setprio(0);
        }
        __syncthreads();   // every wave has read V; the next K is visible
        if (has_next) ld.store_v(Vs, wave, lane);
    }

    // Inputs the bf16 parts do not hold show in the result; such a unit is
    // computed again in f32.
    float down = kPartDown;   // what a result is to be multiplied with
    if (__builtin_amdgcn_ballot_w64(q_code > kQueryCodes || !finite(o)) != 0) {
        unit_f32<D, NB, CAUSAL, VEC>(p, head, unit, t0, min(t1, wave_tiles), 0, o, m_run, l_run);
        down = 1.f;
    }

    float l_tot = pair_sum(l_run);
    if constexpr (SPLIT) {
        if (n_parts > 1) {
            // Partial record of this chunk, lane-major so that every store and
            // load is one coalesced wave access: O^T registers at
            // ws[grid*512 + ((slot*4 + wave)*(D/2) + i)*64 + lane] and
            // (max, sum) at ws[((slot*4 + wave)*64 + lane)*2], slot = pair.
            const int item = head * p.n_wg + wgi;
            const int64_t o_base = (int64_t)gridDim.x * 512;
            {
                float* wo = p.ws + o_base + ((int64_t)pair * 4 + wave) * (D / 2) * 64 + lane;
#pragma unroll
                for (int b = 0; b < NB; ++b)
#pragma unroll
                    for (int r = 0; r < 16; ++r) store_coherent(wo + (b * 16 + r) * 64, o[b][r] * down);
                float* wml = p.ws + (((int64_t)pair * 4 + wave) * 64 + lane) * 2;
                store_coherent(wml, m_run);
                store_coherent(wml + 1, l_tot);
            }
            wait_stores_performed();
            __shared__ unsigned arrival_s;
            __syncthreads();
            if (tid == 0)
                arrival_s = __hip_atomic_fetch_add(p.cnt + item, 1u, __ATOMIC_RELAXED,
                                                   __HIP_MEMORY_SCOPE_AGENT);
            __syncthreads();
            if (arrival_s != (unsigned)(n_parts - 1)) break;   // not the last chunk (uniform)
            if (tid == 0) __hip_atomic_store(p.cnt + item, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);

            // Last chunk: fold the item's records, this one's included, in
            // chunk order (online-softmax combine, GRP records per round
            // trip), so the result does not depend on which chunk came last.
            constexpr int GRP = D >= 128 ? 2 : 4;
            float M = kNegInf;
            l_tot = 0.f;
            down = 1.f;
#pragma unroll
            for (int b = 0; b < NB; ++b)
#pragma unroll
                for (int r = 0; r < 16; ++r) o[b][r] = 0.f;
            const int slot0 = pair - chunk;
            for (int i = 0; i < n_parts; i += GRP) {
                float mc[GRP], lc[GRP], oc[GRP][D / 2];
#pragma unroll
                for (int u = 0; u < GRP; ++u) {
                    // A missing last record of a group reads this chunk's own
                    // record again and is not combined.
                    const int64_t sl = ((int64_t)(slot0 + (i + u < n_parts ? i + u : chunk)) * 4 + wave);
                    const float* ro = p.ws + o_base + sl * (D / 2) * 64 + lane;
                    const float* rml = p.ws + (sl * 64 + lane) * 2;
                    mc[u] = load_coherent(rml);
                    lc[u] = load_coherent(rml + 1);
#pragma unroll
                    for (int e = 0; e < D / 2; ++e) oc[u][e] = load_coherent(ro + e * 64);
                }
#pragma unroll
                for (int u = 0; u < GRP; ++u) {
                    if (i + u >= n_parts) break;
                    const float m_new = fmaxf(M, mc[u]);
                    const float mu = m_new == kNegInf ? 0.f : m_new;
                    const float a = fast_exp2(M - mu), bw = fast_exp2(mc[u] - mu);
                    l_tot = l_tot * a + lc[u] * bw;
#pragma unroll
                    for (int b = 0; b < NB; ++b)
#pragma unroll
                        for (int r = 0; r < 16; ++r) o[b][r] = o[b][r] * a + oc[u][b * 16 + r] * bw;
                    M = m_new;
                }
            }
        }
    }

    // ---- normalise and write O[qrow][dim], dim = 32b + 8(r/4) + 4*half + r%4 --
    const float inv = l_tot > 0.f ? down / l_tot : 0.f;
    if (active && qrow < p.Tq) {
        float* op = p.o.p + bi * p.o.sb + hq * p.o.sh + (int64_t)qrow * p.o.st;
#pragma unroll
        for (int b = 0; b < NB; ++b) {
#pragma unroll
            for (int qq = 0; qq < 4; ++qq) {
                const int c = 32 * b + 8 * qq + 4 * half;
                if (VEC) {
                    if (c < p.d)
                        *reinterpret_cast<float4*>(op + c) =
                            make_float4(o[b][4 * qq] * inv, o[b][4 * qq + 1] * inv,
                                        o[b][4 * qq + 2] * inv, o[b][4 * qq + 3] * inv);
                } else {
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        if (c + j < p.d) op[(c + j) * p.o.sd] = o[b][4 * qq + j] * inv;
                }
            }
        }
    }
    __syncthreads();   // the next item's first tile reuses the LDS stages
    }
}

// Head dims above 128: NW waves of a workgroup of 8 serve one 32-row unit, each
// with DW of its dims -- Q^T and O^T of DW <= 128 dims are what one wave's
// registers hold -- so a workgroup takes 8 / NW units (the (row block, query
// head) units of one KV head, as at d <= 128), which share every staged and
// split K/V tile.  Per 32-key tile each wave computes the partial S^T over its
// dims, leaves it in LDS, and every wave of the unit adds the NW partials in
// wave order: they hold the same S bit for bit and run the same online softmax;
// then each accumulates its DW dims of O^T = V^T P^T.
//
// One workgroup per CU.  Up to 256 dims K and V have a buffer each, replaced a
// phase apart as in the d <= 128 kernel (two barriers per tile); at 512 a tile
// of either is 98 KB, so both go through one buffer (four barriers).  The low
// parts of Q's last steps stay in LDS.
//
// What bounds it: the barriers.  The waves of a CU run their MFMAs and their
// softmax at the same time; up to 256 dims the parts of K and V are therefore
// computed between the MFMAs of the same wave (d = 256, T = 4096 820 -> 785 us,
// d = 192 1830 -> 1690 us).  The matrix cores are busy 48 % of the cycles at 256
// dims and 34 % at 512 (a staged tile serves only 64 rows there: 8 vector
// instructions per MFMA).  Against the f32 MFMAs: B = 1, H = 16, T = 4096 causal,
// d = 256 1204 -> 775 us, d = 512 2412 -> 1964 us; B = 8, H = 20, T = 1500, d = 192
// 2570 -> 1675 us, at 0.6 to 0.7 of the error against 64 bits.
template <int DW, int NW, bool CAUSAL, bool VEC>
__global__ __launch_bounds__(512, 1) void prefill_wide_kernel(const PrefillParams p) {
    constexpr int D = DW * NW, U = 8 / NW;
    using Tile = SplitTile<D, VEC, 8>;
    constexpr int KP = Tile::K_PLANE;
    constexpr int NB = DW / 32;          // 32-wide output column blocks per wave
    constexpr int NT = DW / 16;          // 16-dim steps of a wave's partial S^T
    constexpr int NQL = 4;               // steps whose low parts of Q are in LDS
    constexpr bool ONE = NW > 2;         // K and V share a buffer
    __shared__ __attribute__((aligned(16))) char lds[(ONE ? 3 : 6) * KP + 8 * 4096 + 8 * NQL * 1024];
    char* const Ks = lds;
    char* const Vs = ONE ? lds : lds + 3 * KP;
    char* const Xs = Vs + 3 * KP;        // partial S^T, 4 KB per wave
    char* const Qs = Xs + 8 * 4096;

    const int x = blockIdx.x & 7, q = blockIdx.x >> 3, S = gridDim.x >> 3;

#pragma nounroll
    for (int j = 0;; ++j) {
    int head = 0, wgi = 0;
    const int st = item_at(p, j, x, q, S, head, wgi);
    if (st == 0) break;
    if (st == 2) continue;
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, half = lane >> 5;
    const int dq = wave / U;             // which DW dims this wave holds
    const int bi = head / p.Hkv, kvh = head % p.Hkv;

    const int unit = wgi * U + wave % U;
    const bool active = unit < p.n_units;
    const int rb = active ? unit / p.G : 0;
    const int g = active ? unit % p.G : 0;
    const int hq = kvh * p.G + g;
    const int row0 = rb * 32;
    const int qrow = row0 + l32;

    const int n_kt = (p.Tk + 31) >> 5;
    int last_unit = wgi * U + U - 1;
    if (last_unit > p.n_units - 1) last_unit = p.n_units - 1;
    const int wg_last_key = last_visible_key(p, last_unit / p.G, CAUSAL);
    int n_tiles = wg_last_key < 0 ? 0 : (wg_last_key >> 5) + 1;
    if (n_tiles > n_kt) n_tiles = n_kt;
    const int wave_last_key = last_visible_key(p, rb, CAUSAL);
    const int wave_tiles = active ? (wave_last_key < 0 ? 0 : (wave_last_key >> 5) + 1) : 0;

    // Q^T: three bf16 parts of Q[qrow][dq*DW + 16t + 8*half + 0..7] * scale*log2(e)
    short8 qf[2][NT], ql[NT - NQL];
    char* const qls = Qs + (wave * NQL * 64 + lane) * 16;
    const float* qp = p.q.p + bi * p.q.sb + hq * p.q.sh + (int64_t)qrow * p.q.st;
    const bool rok = active && qrow < p.Tq;
    uint32_t q_code = 0;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        const int c = dq * DW + 16 * t + 8 * half;
        float x[8];
#pragma unroll
        for (int j = 0; j < 8; j += 4) {
            const float4 t4 = (rok && c + j < p.d) ? *reinterpret_cast<const float4*>(qp + c + j)
                                                   : make_float4(0.f, 0.f, 0.f, 0.f);
            x[j] = t4.x; x[j + 1] = t4.y; x[j + 2] = t4.z; x[j + 3] = t4.w;
        }
        uint4 h, m, l;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            x[j] *= p.qscale;
            q_code = max(q_code, range_code(x[j]));
        }
        split3(x[0], x[1], h.x, m.x, l.x);
        split3(x[2], x[3], h.y, m.y, l.y);
        split3(x[4], x[5], h.z, m.z, l.z);
        split3(x[6], x[7], h.w, m.w, l.w);
        qf[0][t] = __builtin_bit_cast(short8, h);
        qf[1][t] = __builtin_bit_cast(short8, m);
        if (t < NT - NQL) ql[t < NT - NQL ? t : 0] = __builtin_bit_cast(short8, l);
        else *reinterpret_cast<uint4*>(qls + (t - (NT - NQL)) * 1024) = l;
    }
    // A query whose parts lose bits makes every S of its row NaN, so that all
    // waves of the unit see it in their results.
    if (q_code > kQueryCodes) qf[0][0] = short8{0x7fc0, 0x7fc0, 0x7fc0, 0x7fc0, 0x7fc0, 0x7fc0, 0x7fc0, 0x7fc0};

    const float* kb = p.k.p + bi * p.k.sb + kvh * p.k.sh;
    const float* vb = p.v.p + bi * p.v.sb + kvh * p.v.sh;

    floatx16 o[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[b][r] = 0.f;
    float m_run = kNegInf, l_run = 0.f;

    // Second items of causal pairs walk their key tiles backwards, as in the
    // d <= 128 kernel (a head's K/V tiles stay in the XCD's L2: 688 -> 260 MB
    // read at B = 1, H = 16, T = 4096, d = 256 on the f32 MFMAs; 292 now).
    const bool rev = p.pairing && (j & 1);
    const int kstep = rev ? -1 : 1;
    const int kfirst = rev ? n_tiles - 1 : 0;
    Tile ld;
    ld.init(p, wave, lane);
    if (n_tiles > 0) {
        ld.load_k(p, kb, kfirst * 32, wave, lane, true);
        ld.load_v(p, vb, kfirst * 32, wave, lane, true);
        ld.store_k(Ks, wave, lane);
    }
    __syncthreads();

    for (int it = 0; it < n_tiles; ++it) {
        const int kt = kfirst + kstep * it;
        const bool has_next = it + 1 < n_tiles;
        const bool mine = kt < wave_tiles;
        floatx16 s;
        const float m_use = (m_run == kNegInf) ? 0.f : m_run;
        if (mine) {
            // Partial S^T = K Q^T over this wave's dims, log2 domain.
#pragma unroll
            for (int r = 0; r < 16; ++r) s[r] = 0.f;
            const char* kw = Ks + dq * NT * 1024;
            __builtin_amdgcn_s_setprio(1);
            // The operands of a step are read one step ahead; between the later
            // steps (its loads are still under way before) this tile's V is
            // split, which no other wave of the SIMD would hide: all of a
            // workgroup's waves run their MFMAs at the same time.
            short8 kc[3], kn[3];
            const auto read_k = [&](int t, short8* f) {
                const char* a = kw + t * 1024 + half * 512 + ((l32 ^ ((2 * (dq * NT + t) + half) & 15)) << 4);
                f[0] = *reinterpret_cast<const short8*>(a);
                f[1] = *reinterpret_cast<const short8*>(a + KP);
                f[2] = *reinterpret_cast<const short8*>(a + 2 * KP);
            };
            read_k(0, kc);
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                short8 qlt;
                if (t < NT - NQL) qlt = ql[t < NT - NQL ? t : 0];
                else qlt = *reinterpret_cast<const short8*>(qls + (t - (NT - NQL)) * 1024);
                if (t + 1 < NT) read_k(t + 1, kn);
                s = mfma_bf16(kc[2], qf[0][t], s);
                s = mfma_bf16(kc[1], qf[1][t], s);
                s = mfma_bf16(kc[1], qf[0][t], s);
                s = mfma_bf16(kc[0], qf[1][t], s);
                s = mfma_bf16(kc[0], qlt, s);
                if (!ONE) {
#pragma unroll
                    for (int i = 0; i < 4 * Tile::NJ; ++i)
                        if (NT / 2 + i * (NT / 2) / (4 * Tile::NJ) == t) ld.part_v(i, Vs, wave, lane);
                }
#pragma unroll
                for (int u = 0; u < 3; ++u) kc[u] = kn[u];
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                const char* a = kw + t * 1024 + half * 512 + ((l32 ^ ((2 * (dq * NT + t) + half) & 15)) << 4);
                s = mfma_bf16(*reinterpret_cast<const short8*>(a), qf[0][t], s);
            }
            __builtin_amdgcn_s_setprio(0);
            // This wave's partial, register-group major (each store one
            // contiguous, conflict-free 1 KB wave access).
            char* xo = Xs + wave * 4096 + lane * 16;
#pragma unroll
            for (int i = 0; i < 4; ++i)
                *reinterpret_cast<float4*>(xo + 1024 * i) =
                    make_float4(s[4 * i], s[4 * i + 1], s[4 * i + 2], s[4 * i + 3]);
        } else if (!ONE) {
            ld.store_v(Vs, wave, lane);
        }
        if (!ONE) ld.load_k(p, kb, (kt + kstep) * 32, wave, lane, has_next);
        __syncthreads();   // partials visible, K read (and V visible)
        if (ONE) {
            ld.store_v(Vs, wave, lane);
            ld.load_k(p, kb, (kt + kstep) * 32, wave, lane, has_next);
        }
        if (mine) {
            // S^T - m: the unit's partials in wave order.
            const char* xi = Xs + (wave % U) * 4096 + lane * 16;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                float4 a = *reinterpret_cast<const float4*>(xi + 1024 * i);
#pragma unroll
                for (int w = 1; w < NW; ++w) {
                    const float4 t = *reinterpret_cast<const float4*>(xi + w * U * 4096 + 1024 * i);
                    a.x += t.x; a.y += t.y; a.z += t.z; a.w += t.w;
                }
                s[4 * i] = a.x - m_use; s[4 * i + 1] = a.y - m_use;
                s[4 * i + 2] = a.z - m_use; s[4 * i + 3] = a.w - m_use;
            }
            const int key0 = kt * 32;
            const bool need_mask = (key0 + 32 > p.Tk) || (CAUSAL && key0 + 31 > row0 + p.q_offset);
            if (need_mask) {
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int key = key0 + 8 * (r >> 2) + 4 * half + (r & 3);
                    const bool vis = key < p.Tk && (!CAUSAL || key <= qrow + p.q_offset);
                    s[r] = vis ? s[r] : kNegInf;
                }
            }
            // Online softmax with the lazy rescale of the d <= 128 kernel; all
            // waves of the unit take the same decisions on the same values.
            float mt = s[0];
#pragma unroll
            for (int r = 1; r < 16; ++r) mt = fmaxf(mt, s[r]);
            mt = pair_max(mt);
            if (__builtin_amdgcn_ballot_w64(mt > (m_run == kNegInf ? kNegInf : 8.f)) != 0) {
                const float m_new = fmaxf(m_run, mt + m_use);
                const float n_use = (m_new == kNegInf) ? 0.f : m_new;
                const float alpha = fast_exp2(m_run - n_use);
                l_run *= alpha;
#pragma unroll
                for (int b = 0; b < NB; ++b)
#pragma unroll
                    for (int r = 0; r < 16; ++r) o[b][r] *= alpha;
#pragma unroll
                for (int r = 0; r < 16; ++r) s[r] -= n_use - m_use;
                m_run = m_new;
            }
            float ls = 0.f;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                s[r] = fast_exp2(s[r]);
                ls += s[r];
            }
            l_run += ls;
        }
        if (ONE) __syncthreads();   // V visible
        if (mine) {
            // O^T += V^T P^T over this wave's output dims, the next K split
            // between the MFMAs.
            uint32_t pp[2][3][4];
            const auto part_p = [&](int i) {
                split3(s[2 * i] * kPartUp, s[2 * i + 1] * kPartUp, pp[i >> 2][0][i & 3], pp[i >> 2][1][i & 3],
                       pp[i >> 2][2][i & 3]);
            };
            const auto operand = [&](int st, int u) {
                return __builtin_bit_cast(short8, make_uint4(pp[st][u][0], pp[st][u][1], pp[st][u][2], pp[st][u][3]));
            };
            short8 vc[3], vn[3];
            const auto read_v = [&](int i, short8* f) {
                const char* a = Vs + (((dq * NB + i % NB) * 2 + i / NB) * 64 + lane) * 16;
                f[0] = *reinterpret_cast<const short8*>(a);
                f[1] = *reinterpret_cast<const short8*>(a + KP);
                f[2] = *reinterpret_cast<const short8*>(a + 2 * KP);
            };
            if (!ONE) read_v(0, vc);   // (read ahead: 12 registers that 512 dims do not have)
#pragma unroll
            for (int i = 0; i < 4; ++i) part_p(i);
            __builtin_amdgcn_s_setprio(1);
#pragma unroll
            for (int i = 0; i < 2 * NB; ++i) {
                const int b = i % NB, st = i / NB;
                if (ONE) read_v(i, vc);
                else if (i + 1 < 2 * NB) read_v(i + 1, vn);
                const short8 ph = operand(st, 0), pm = operand(st, 1), pl = operand(st, 2);
                o[b] = mfma_bf16(vc[2], ph, o[b]);
                o[b] = mfma_bf16(vc[0], pl, o[b]);
                o[b] = mfma_bf16(vc[1], pm, o[b]);
                o[b] = mfma_bf16(vc[1], ph, o[b]);
                o[b] = mfma_bf16(vc[0], pm, o[b]);
                o[b] = mfma_bf16(vc[0], ph, o[b]);
                if (st == 0) {
#pragma unroll
                    for (int u = 4 + 4 * b / NB; u < 4 + 4 * (b + 1) / NB; ++u) part_p(u);
                }
                if (!ONE) {
#pragma unroll
                    for (int u = i * Tile::NK / (2 * NB); u < (i + 1) * Tile::NK / (2 * NB); ++u)
                        ld.part_k(u, Ks, wave, lane);
                }
                if (!ONE) {
#pragma unroll
                    for (int u = 0; u < 3; ++u) vc[u] = vn[u];
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            __builtin_amdgcn_s_setprio(0);
        } else if (!ONE) {
            ld.store_k(Ks, wave, lane);
        }
        if (!ONE) ld.load_v(p, vb, (kt + kstep) * 32, wave, lane, has_next);
        __syncthreads();   // V and the partials are read (and the next K visible)
        if (ONE) {
            if (has_next) ld.store_k(Ks, wave, lane);
            ld.load_v(p, vb, (kt + kstep) * 32, wave, lane, has_next);
            __syncthreads();   // the next K is visible
        }
    }

    float down = kPartDown;
    if (__builtin_amdgcn_ballot_w64(!finite(o)) != 0) {
        unit_f32<D, NB, CAUSAL, true>(p, head, unit, 0, wave_tiles, dq * DW, o, m_run, l_run);
        down = 1.f;
    }

    const float l_tot = pair_sum(l_run);
    const float inv = l_tot > 0.f ? down / l_tot : 0.f;
    if (active && qrow < p.Tq) {
        float* op = p.o.p + bi * p.o.sb + hq * p.o.sh + (int64_t)qrow * p.o.st;
#pragma unroll
        for (int b = 0; b < NB; ++b) {
#pragma unroll
            for (int qq = 0; qq < 4; ++qq) {
                const int c = dq * DW + 32 * b + 8 * qq + 4 * half;
                if (c < p.d)
                    *reinterpret_cast<float4*>(op + c) =
                        make_float4(o[b][4 * qq] * inv, o[b][4 * qq + 1] * inv,
                                    o[b][4 * qq + 2] * inv, o[b][4 * qq + 3] * inv);
            }
        }
    }
    __syncthreads();   // the next item's first tile reuses the LDS stages
    }
}

// CUs and resident workgroups per CU of the kernel on the current device.
template <int D, bool CAUSAL, bool VEC>
void residency(int& cus, int& per_cu) {
    constexpr auto kernel = prefill_mfma_kernel<D, CAUSAL, VEC, false>;
    // Atomic: callers on several threads may fill the cache at once.
    static std::atomic<int> cached_cus[64], cached_per[64];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) dev = 0;
    int c = cached_cus[dev].load(std::memory_order_acquire);
    int k = cached_per[dev].load(std::memory_order_relaxed);
    if (c == 0 || k == 0) {
        if (hipDeviceGetAttribute(&c, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || c < 8) c = 256;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&k, kernel, 256, 0) !=
                hipSuccess || k < 1)
            k = 1;
        cached_per[dev].store(k, std::memory_order_relaxed);
        cached_cus[dev].store(c, std::memory_order_release);
    }
    cus = c;
    per_cu = k;
}

int device_cus() {
    static std::atomic<int> cached[64];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) dev = 0;
    int c = cached[dev].load(std::memory_order_relaxed);
    if (c == 0) {
        if (hipDeviceGetAttribute(&c, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || c < 8)
            c = 256;
        cached[dev].store(c, std::memory_order_relaxed);
    }
    return c;
}

// One resident wave of persistent workgroups: k per CU on every CU (an
// uneven count would leave the CUs that hold more workgroups behind), 8*S in
// all with S = k * CUs / 8 per XCD, each XCD's super-items dealt round-robin.
// k minimises rounds * k (the time of a round grows with the workgroups that
// share a CU; one workgroup per CU leaves its SIMDs a single wave, taken as
// 30 % slower).  Causal problems with enough work pair ranks r and n_wg-1-r
// so that every super-item costs the same.  Fills p's schedule fields and
// returns S.
int persistent_slots(PrefillParams& p, bool causal, int cus, int k_max) {
    const int cu_per_xcd = cus / 8;
    const int64_t heads = (int64_t)p.B * p.Hkv;
    p.pairing = (causal && p.n_wg > 1 && heads * ((p.n_wg + 1) / 2) >= (int64_t)cus * k_max) ? 1 : 0;
    p.n_pairs = p.pairing ? (p.n_wg + 1) / 2 : p.n_wg;
    p.n_super = (int)(heads * p.n_pairs);
    p.per_xcd = (p.n_super + 7) / 8;
    int S = 1, best_rounds = 1;
    double best = 1e300;
    for (int k = 1; k <= k_max; ++k) {
        const int s = k * cu_per_xcd;
        const int rounds = (p.per_xcd + s - 1) / s;
        const double cost = (double)rounds * k * (k == 1 ? 1.3 : 1.0);
        if (cost < best) { best = cost; S = s; best_rounds = rounds; }
    }
    // A partly empty last round costs more than the hardware's own dispatch of
    // one super-item per workgroup (which also covers small problems).
    if (S >= p.per_xcd || (double)p.per_xcd / ((double)best_rounds * S) < 0.97) S = p.per_xcd;
    // Hardware dispatch of unpaired causal items: in head-major rank order the
    // two workgroups placed on a CU take items of the same rank from two heads
    // (both long or both short).  Longest first across the XCD's heads, with
    // complementary lengths per CU, took B = 1, H = 16, T = 4096, d = 128 from
    // 1016 to 592 us and B = 1, Hq = 32, Hkv = 8, T = 2048 from 401 to 296 us.
    p.order_cu = 0;
    p.order_hpx = 0;
    p.order_all = 0;
    // One workgroup per CU and more items than CUs: the order above would give the
    // CUs that finish first the shortest items left and leave the longest running
    // alone, and pairs that do not fill their last round idle up to half the CUs.
    // All heads' items, longest first, as CUs get free (us; the deep kernel): d =
    // 320, 14 heads, T = 2300 743 -> 442 (679), 17 heads, T = 1024 231 -> 183 (220), 2 KV
    // heads of 16, T = 700 216 -> 128 (205); d = 192, 48 heads, T = 1500 440 -> 284, 9
    // heads, T = 6000 1258 -> 800.  Pairs that fill their rounds keep a head's K/V in
    // one XCD's L2: d = 512, 16 heads, T = 2048 493 against 505.
    const int64_t items = heads * p.n_wg;
    if (causal && k_max == 1 && items > cus && items < INT32_MAX - 8 &&
        (!p.pairing || (double)p.per_xcd / ((double)((p.per_xcd + cu_per_xcd - 1) / cu_per_xcd) * cu_per_xcd) < 0.9)) {
        p.pairing = 0;
        p.order_all = 1;
        return (int)((items + 7) / 8);
    }
    if (causal && !p.pairing && S == p.per_xcd && heads % 8 == 0 && cu_per_xcd > 0 &&
        (int64_t)p.per_xcd * 8 == heads * p.n_wg) {
        p.order_cu = cu_per_xcd;
        p.order_hpx = (int)(heads / 8);
    }
    return S;
}

template <int D, bool CAUSAL, bool VEC>
hipError_t launch_t(PrefillParams p, hipStream_t stream) {
    if (p.n_chunks > 1 && p.ws && p.cnt) {
        hipLaunchKernelGGL((prefill_mfma_kernel<D, CAUSAL, VEC, true>),
                           dim3(8 * ((p.B * p.Hkv * p.part_prefix[p.n_wg] + 7) / 8)), dim3(256), 0, stream, p);
        return hipGetLastError();
    }
    int cus = 0, k_max = 0;
    residency<D, CAUSAL, VEC>(cus, k_max);
    const int S = persistent_slots(p, CAUSAL, cus, k_max);
    hipLaunchKernelGGL((prefill_mfma_kernel<D, CAUSAL, VEC, false>), dim3(8 * S), dim3(256), 0, stream, p);
    return hipGetLastError();
}

// Head dims 129..512: one workgroup of 8 waves per CU.
template <int DW, int NW, bool VEC = true>
hipError_t launch_wide_d(PrefillParams p, bool causal, hipStream_t stream) {
    constexpr int U = 8 / NW;
    p.n_wg = (p.n_units + U - 1) / U;
    p.total = p.B * p.Hkv * p.n_wg;
    const int S = persistent_slots(p, causal, device_cus(), 1);
    if (causal)
        hipLaunchKernelGGL((prefill_wide_kernel<DW, NW, true, VEC>), dim3(8 * S), dim3(512), 0, stream, p);
    else
        hipLaunchKernelGGL((prefill_wide_kernel<DW, NW, false, VEC>), dim3(8 * S), dim3(512), 0, stream, p);
    return hipGetLastError();
}

template <int D>
hipError_t launch_d(const PrefillParams& p, bool causal, bool vec, hipStream_t stream) {
    if (causal) return vec ? launch_t<D, true, true>(p, stream) : launch_t<D, true, false>(p, stream);
    return vec ? launch_t<D, false, true>(p, stream) : launch_t<D, false, false>(p, stream);
}

}  // namespace

int prefill_padded_dim(int d) {
    if (d <= 32) return 32;
    if (d <= 64) return 64;
    if (d <= 128) return 128;
    return 0;
}

namespace {

void derive_schedule(PrefillParams& p) {
    p.G = p.Hq / p.Hkv;
    p.n_rb = (p.Tq + 31) / 32;
    p.n_units = p.G * p.n_rb;
    p.n_wg = (p.n_units + 3) / 4;
    p.total = p.B * p.Hkv * p.n_wg;
}

}  // namespace

// A problem with fewer work items than CUs leaves most SIMDs idle, and its
// time is the longest item's chain of key tiles.  Cutting every item's tiles
// into chunks, sized so that the chunks fill the CUs once (at most 16 chunks
// per item), shortens that chain to one chunk plus the merge of the item's
// records.
PrefillSplit prefill_split_plan(PrefillParams& p, bool causal, bool vec) {
    (void)vec;
    PrefillSplit r{0, 0};
    p.n_chunks = 0;
    p.chunk_tiles = 0;
    derive_schedule(p);
    const int D = prefill_padded_dim(p.d);
    const int cus = device_cus();
    if (p.total == 0 || D == 0 || p.total >= cus || p.n_wg > kMaxSplitItems) return r;
    // Key tiles of each work item, as the kernel counts them.
    const int n_kt = (p.Tk + 31) / 32;
    std::vector<int> tiles(p.n_wg);
    int max_t = 0;
    for (int w = 0; w < p.n_wg; ++w) {
        const int last_unit = std::min(w * 4 + 3, p.n_units - 1);
        int lk = p.Tk - 1;
        if (causal) {
            const int last_row = std::min(last_unit / p.G * 32 + 31, p.Tq - 1);
            lk = std::min(last_row + p.q_offset, p.Tk - 1);
        }
        tiles[w] = lk < 0 ? 0 : std::min(lk / 32 + 1, n_kt);
        max_t = std::max(max_t, tiles[w]);
    }
    if (max_t < 4) return r;
    // The chunk of the least cost by a model fitted to 1300 measured calls (11 to 160
    // key tiles, 1 to 16 heads; within 3 % rms at one workgroup per CU, 7 % at two):
    // a start, the tiles of a chunk one after the other, and a record per part for
    // the last chunk to fold.  Two workgroups on a CU share its matrix cores but
    // fill each other's waits; three were slower throughout.  Measured (us, by
    // chunk tiles): d = 128, one head, T = 512 26.9 [1], 23.3 [2], 26.0 [4]; 8 heads,
    // T = 300 21.4 [1], 20.3 [2], 22.7 [3]; 32 heads over 8, T = 509 35.6 [3], 32.9
    // [6], 35.4 [7]; 16 over 4, B = 2, 333 rows over 3001 keys 118 [10], 103 [18], 139
    // [40]; d = 32, the same 42.8 [7], 37.4 [12], 59.4 [43].
    // Candidates: the shortest chunk of each number of parts (at most 16 per item),
    // and the shortest that leaves one or two workgroups per CU.
    struct Cost { double tile, start, part; };   // us
    static constexpr Cost kCost[3][2] = {{{1.2, 6.2, 0.32}, {1.4, 7.2, 0.46}},
                                         {{1.8, 7.8, 0.52}, {2.1, 10.1, 0.73}},
                                         {{3.0, 9.7, 0.94}, {3.7, 14.2, 1.33}}};
    const Cost* cost = kCost[D == 32 ? 0 : D == 64 ? 1 : 2];
    const auto workgroups = [&](int c) {
        int64_t n = 0;
        for (int t : tiles) n += std::max(1, (t + c - 1) / c);
        return n * p.B * p.Hkv;
    };
    int ch = max_t;
    double best = 1e300;
    const auto consider = [&](int c) {
        const int64_t n = workgroups(c);
        if (n > 2 * (int64_t)cus) return;
        const Cost& k = cost[n > cus];
        const double us = k.tile * c + k.start + k.part * ((max_t + c - 1) / c);
        if (us < best) { best = us; ch = c; }
    };
    for (int m = 1; m <= 16; ++m) consider((max_t + m - 1) / m);
    for (int k = 1; k <= 2; ++k) {
        int lo = (max_t + 15) / 16, hi = max_t;
        while (lo < hi) {
            const int mid = (lo + hi) / 2;
            if (workgroups(mid) <= (int64_t)k * cus) hi = mid;
            else lo = mid + 1;
        }
        consider(lo);
    }
    const int nc = (max_t + ch - 1) / ch;
    if (nc < 2) return r;
    p.n_chunks = nc;
    p.chunk_tiles = ch;
    p.part_prefix[0] = 0;
    for (int w = 0; w < p.n_wg; ++w)
        p.part_prefix[w + 1] = (uint16_t)(p.part_prefix[w] + std::max(1, (tiles[w] + ch - 1) / ch));
    // Per workgroup: (max, sum) of 4 waves x 64 lanes, and 4 x D/2 x 64 O values.
    const uint64_t grid = ((uint64_t)p.B * p.Hkv * p.part_prefix[p.n_wg] + 7) / 8 * 8;
    r.ws_bytes = grid * (512 + 128 * (uint64_t)D) * 4;
    r.n_counters = p.total;
    return r;
}

// The vector loads of a K/V tile hold its row offsets in 32 bits.
static bool row_offsets_fit(const PrefillParams& p) {
    return p.k.st >= 0 && p.k.st < kMaxTileStride && p.v.st >= 0 && p.v.st < kMaxTileStride;
}

hipError_t launch_prefill_wide(PrefillParams p, bool causal, hipStream_t stream) {
    derive_schedule(p);
    if (p.total == 0) return hipSuccess;
    if (p.d <= 128 || p.d > 512) return hipErrorInvalidValue;
    if (!row_offsets_fit(p))
        return p.d <= 256 ? launch_wide_d<128, 2, false>(p, causal, stream) : hipErrorInvalidValue;
    if (p.d <= 192) return launch_wide_d<96, 2>(p, causal, stream);
    if (p.d <= 256) return launch_wide_d<128, 2>(p, causal, stream);
    if (p.d <= 384) return launch_wide_d<96, 4>(p, causal, stream);
    return launch_wide_d<128, 4>(p, causal, stream);
}

hipError_t launch_prefill(PrefillParams p, bool causal, bool vec, hipStream_t stream) {
    derive_schedule(p);
    if (p.total == 0) return hipSuccess;
    vec = vec && row_offsets_fit(p);
    switch (prefill_padded_dim(p.d)) {
        case 32: return launch_d<32>(p, causal, vec, stream);
        case 64: return launch_d<64>(p, causal, vec, stream);
        case 128: return launch_d<128>(p, causal, vec, stream);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace nne
