// The hidden stack and head of mlp_tile.hpp for a tile of 16 rows instead of 32:
// v_mfma_f32_16x16x4_f32, each wavefront owning NT tiles of 16 output columns.
//
// The fp32 matrix instructions accumulate their k products as one serial chain of fused
// multiply-adds in ascending k, whatever the tile shape, so with the k-steps taken in ascending
// order this tile gives the same bits as the 32-row tile (and as a serial fmaf loop): a kernel may
// pick the tile height that suits its launch without changing results.
//
// Operand layout of v_mfma_f32_16x16x4_f32, lane = 16 g + n:
//   A[row n][k g], B[k g][column n]  ->  D[row 4 g + v][column n], v = 0 .. 3.
// The columns of a wavefront start at c0; its first four tiles interleave (tile q holds columns
// c0 + 4 n + q), so that one 16-byte load per k-step fetches the B operands of all four from one
// contiguous 256-byte run of the weight row; a fifth tile holds c0 + 64 + n, a fifth and sixth
// together c0 + 64 + 2 n + (q - 4), one 8-byte load.
#pragma once
#include "mlp_tile.hpp"

namespace mrl {

typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int PR16 = 16;            // rows per tile
constexpr int HT16_LD = PR16 + 1;   // k-major activations hT[k][row]

template <int NT>
MRL_DEV int tile16_col(int c0, int q, int n) {
    static_assert(NT >= 1 && NT <= 6, "one to six column tiles per wavefront");
    if (NT <= 4 || q < 4) return c0 + (NT >= 4 ? 4 * n + q : NT * n + q);
    return NT == 5 ? c0 + 64 + n : c0 + 64 + 2 * n + (q - 4);
}

// The observations of a block's 16 envs, `at(row, column)`, into xs and out to the rollout row; rows beyond `ne` are zero.
// (Straight-line: ahead of a loop with stores the compiler waits for every load in flight, here the weights':
// LunarLander, hidden width 256, 8192 envs 28.7 : 27.3 us per step, width 64, 4096 envs 11.36 : 11.18.)
template <int IN, int T, class At>
MRL_DEV void stage_observations(float *xs, float *r_obs, int ne, int tid, At &&at) {
#pragma unroll
    for (int q = 0; q < (PR16 * IN + T - 1) / T; ++q) {
        const int i = tid + q * T, r = i / IN, c = i - r * IN;
        if (r < PR16) {
            float v = 0.0f;
            if (r < ne) {
                v = at(r, c);
                r_obs[i] = v;
            }
            xs[r * XS_LD + c] = v;
        }
    }
}

// a pointer that is the same in all lanes of a wavefront, in scalar registers
MRL_DEV const float *wave_uniform(const float *p) {
    const uint64_t u = reinterpret_cast<uint64_t>(p);
    const uint32_t lo = __builtin_amdgcn_readfirstlane((int)(uint32_t)u), hi = __builtin_amdgcn_readfirstlane((int)(u >> 32));
    return reinterpret_cast<const float *>((uint64_t)hi << 32 | lo);
}

// Where a lane's operands of a weight row lie: byte offsets from the row's start, which stays a scalar.
template <int NT>
struct Tile16Lane {
    uint32_t o, ox;
    MRL_DEV Tile16Lane(int H, int c0, int lane) {
        const int g = lane >> 4, n = lane & 15, col = g * H + c0;
        o = 4u * (uint32_t)(col + (NT >= 4 ? 4 : NT) * n);
        ox = 4u * (uint32_t)(col + 64 + (NT == 5 ? 1 : 2) * n);
    }
    // ahead of a block's loads: the widening of the offsets stays beside them, where it folds into the address mode
    MRL_DEV void here() { asm("" : "+v"(o), "+v"(ox)); }
    MRL_DEV void load(const float *row, float (&b)[NT]) const {
        typedef const char __attribute__((address_space(1))) *Row;
        Row r = (Row)(reinterpret_cast<const char *>(row));
        asm("" : "+s"(r));   // (not folded into the lanes' offsets, which would make every address a 64-bit vector sum)
        if constexpr (NT >= 4) {
            const floatx4 v = *(const floatx4 __attribute__((address_space(1))) *)(r + o);
#pragma unroll
            for (int q = 0; q < 4; ++q) b[q] = v[q];
            if constexpr (NT == 5) b[4] = *(const float __attribute__((address_space(1))) *)(r + ox);
            if constexpr (NT == 6) {
                const floatx2 x = *(const floatx2 __attribute__((address_space(1))) *)(r + ox);
                b[4] = x[0]; b[5] = x[1];
            }
        } else {
#pragma unroll
            for (int q = 0; q < NT; ++q) b[q] = *(const float __attribute__((address_space(1))) *)(r + o + 4 * q);
        }
    }
};

// Row-independent operands of the hidden stack (biases, layer-0 weights, first block of layer-1
// weights), requested before the tile's rows are staged.  IN = input width (compile time here).
template <int H, int IN, int NT, int KB>
struct Hidden16Operands {
    static constexpr int K0 = (IN + 3) / 4;
    float bias0[NT], bias1[NT];
    float w0[K0][NT];
    float bv[KB][NT];
    MRL_DEV void load(const float *__restrict__ p, int c0, int lane) {
        const int g = lane >> 4;
        const float *W0 = wave_uniform(p), *b0 = W0 + IN * H;
        const float *W1 = b0 + H, *b1 = W1 + H * H;
        Tile16Lane<NT> row(0, c0, lane), at(H, c0, lane);   // (a bias "matrix" is one row)
        row.here();
        at.here();
        row.load(b0, bias0);
        row.load(b1, bias1);
#pragma unroll
        for (int kk = 0; kk < K0; ++kk) {
            if (IN % 4 == 0 || 4 * kk + g < IN) {
                at.load(W0 + 4 * kk * H, w0[kk]);
            } else {
#pragma unroll
                for (int q = 0; q < NT; ++q) w0[kk][q] = 0.0f;
            }
        }
#pragma unroll
        for (int j = 0; j < KB; ++j) at.load(W1 + 4 * j * H, bv[j]);
    }
};

// Layer 0 of a tile: a0[kk] = input 4 kk + g of row n, hT [H][HT16_LD] receives act(layer 0) k-major.
template <int H, int IN, int ACT, int NT, int KB>
MRL_DEV void hidden16_layer0_of(const float (&a0)[(IN + 3) / 4], float *hT, const Hidden16Operands<H, IN, NT, KB> &ops, int c0, int lane) {
    constexpr int K0 = (IN + 3) / 4;
    const int g = lane >> 4, n = lane & 15;
    floatx4 c[NT];
#pragma unroll
    for (int q = 0; q < NT; ++q) c[q] = floatx4{0};
#pragma unroll
    for (int kk = 0; kk < K0; ++kk) {
#pragma unroll
        for (int q = 0; q < NT; ++q)
            c[q] = __builtin_amdgcn_mfma_f32_16x16x4f32(a0[kk], ops.w0[kk][q], c[q], 0, 0, 0);
    }
#pragma unroll
    for (int q = 0; q < NT; ++q) {
        const int col = tile16_col<NT>(c0, q, n);
#pragma unroll
        for (int v = 0; v < 4; ++v) hT[col * HT16_LD + 4 * g + v] = activate<ACT>(c[q][v] + ops.bias0[q]);
    }
}
// the same from xs[16][XS_LD]
template <int H, int IN, int ACT, int NT, int KB>
MRL_DEV void hidden16_layer0(const float *xs, float *hT, const Hidden16Operands<H, IN, NT, KB> &ops, int c0, int lane) {
    constexpr int K0 = (IN + 3) / 4;
    const int g = lane >> 4, n = lane & 15;
    float a0[K0];
#pragma unroll
    for (int kk = 0; kk < K0; ++kk) {
        const int k = 4 * kk + g;
        a0[kk] = k < IN ? xs[n * XS_LD + k] : 0.0f;
    }
    hidden16_layer0_of<H, IN, ACT, NT, KB>(a0, hT, ops, c0, lane);
}

// Biases and activation of layer 1: h2 [16][H + 1] receives act(c + bias) row-major.
template <int H, int IN, int ACT, int NT, int KB>
MRL_DEV void hidden16_layer1_end(const floatx4 (&c)[NT], float *h2, const Hidden16Operands<H, IN, NT, KB> &ops, int c0, int lane) {
    const int g = lane >> 4, n = lane & 15;
#pragma unroll
    for (int q = 0; q < NT; ++q) {
        const int col = tile16_col<NT>(c0, q, n);
#pragma unroll
        for (int v = 0; v < 4; ++v) h2[(4 * g + v) * (H + 1) + col] = activate<ACT>(c[q][v] + ops.bias1[q]);
    }
}
// k-steps J0 .. J1 - 1 of layer 1 with all its weights held
template <int H, int J0, int J1, int IN, int NT>
MRL_DEV void hidden16_layer1_steps(const float *hT, const Hidden16Operands<H, IN, NT, H / 4> &ops, floatx4 (&c)[NT], int lane) {
    const float *ht = hT + (lane >> 4) * HT16_LD + (lane & 15);
    float a[J1 - J0];
#pragma unroll
    for (int j = J0; j < J1; ++j) a[j - J0] = ht[4 * j * HT16_LD];
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = J0; j < J1; ++j) {
#pragma unroll
        for (int q = 0; q < NT; ++q) c[q] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[j - J0], ops.bv[j][q], c[q], 0, 0, 0);
    }
}

// Layer 1: weights streamed from L2 one block of KB k-steps ahead of the MFMAs (KB = H / 4: all of them are in
// `ops`, which is then left as it is); h2 [16][H + 1] receives act(layer 1) row-major.  before_h2() is called between
// the last read of hT and the first write of h2.  The blocks alternate between two register sets, and a load's
// address is a scalar pair and a 32-bit lane offset: with one set copied to the other, the copies at a block's start
// waited for its last load, and with 64-bit vector addresses they were 129 instructions beside the 40 MFMAs of a
// five-tile block (now 56), on a SIMD that issues one or the other.  us per rollout step before : now, hidden width 256:
// LunarLander 4096 envs 21.2 : 19.2, 8192 envs 31.5 : 29.2, CartPole 1024 envs 13.0 : 10.8; width 128, LunarLander 4096
// envs 14.5 : 13.7.
template <int H, int IN, int ACT, int NT, int KB, class Before>
MRL_DEV void hidden16_layer1(const float *__restrict__ p, const float *hT, float *h2, Hidden16Operands<H, IN, NT, KB> &ops,
                             int c0, int lane, Before &&before_h2) {
    constexpr int NBLK = H / (4 * KB);
    static_assert((H / 4) % KB == 0 && (NBLK == 1 || NBLK % 2 == 0), "whole pairs of blocks of k-steps");
    const int g = lane >> 4, n = lane & 15;
    const float *W1 = p + IN * H + H;
    floatx4 c[NT];
#pragma unroll
    for (int q = 0; q < NT; ++q) c[q] = floatx4{0};
    auto fetch = [&](const float *ht, const float *w, Tile16Lane<NT> &at, float (&a)[KB], float (&b)[KB][NT]) {
        at.here();
#pragma unroll
        for (int j = 0; j < KB; ++j) {
            a[j] = ht[4 * j * HT16_LD];
            at.load(w + 4 * j * H, b[j]);
        }
    };
    auto product = [&](const float (&a)[KB], const float (&b)[KB][NT]) {
        __builtin_amdgcn_sched_barrier(0);   // the loads above stay ahead of these MFMAs
#pragma unroll
        for (int j = 0; j < KB; ++j) {
#pragma unroll
            for (int q = 0; q < NT; ++q) c[q] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[j], b[j][q], c[q], 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    const float *ht = hT + g * HT16_LD + n;
    float a[KB];
#pragma unroll
    for (int j = 0; j < KB; ++j) a[j] = ht[4 * j * HT16_LD];
    if constexpr (NBLK == 1) {
        product(a, ops.bv);
    } else {
        Tile16Lane<NT> at(H, c0, lane);
        W1 = wave_uniform(W1);
        float na[KB], nb[KB][NT];
        constexpr int HT_BLK = 4 * KB * HT16_LD, W_BLK = 4 * KB * H;
        for (int blk = 2; blk < NBLK; blk += 2) {
            fetch(ht + HT_BLK, W1 + W_BLK, at, na, nb);
            product(a, ops.bv);
            fetch(ht + 2 * HT_BLK, W1 + 2 * W_BLK, at, a, ops.bv);
            product(na, nb);
            ht += 2 * HT_BLK;
            W1 += 2 * W_BLK;
        }
        fetch(ht + HT_BLK, W1 + W_BLK, at, na, nb);
        product(a, ops.bv);
        product(na, nb);
    }
    before_h2();
    hidden16_layer1_end<H, IN, ACT, NT, KB>(c, h2, ops, c0, lane);
}

// Hidden stack of one net for the block's 16 rows on the wavefronts that share it (each with its
// own c0 / NT; `lane` = lane of the calling wavefront).  xs[16][XS_LD] holds the inputs, hT
// [H][HT16_LD] receives act(layer 0) k-major, h2 [16][H + 1] act(layer 1) row-major; h2 may share
// its memory with hT (H2_ON_HT: everyone has finished reading hT before h2 is written).  sync() is
// the barrier of the wavefronts that work on this net.
template <int H, int IN, int ACT, int NT, int KB, bool H2_ON_HT, class Sync>
MRL_DEV void hidden_stack16(const float *__restrict__ p, const float *xs, float *hT, float *h2,
                            Hidden16Operands<H, IN, NT, KB> &ops, int c0, int lane, Sync &sync) {
    static_assert(PR16 * (H + 1) <= H * HT16_LD, "h2 fits into hT");
    hidden16_layer0<H, IN, ACT, NT, KB>(xs, hT, ops, c0, lane);
    sync();
    hidden16_layer1<H, IN, ACT, NT, KB>(p, hT, h2, ops, c0, lane, [&]() { if (H2_ON_HT) sync(); });
    sync();
}

// Sum over TPR neighbouring lanes (all of a wavefront's rows of 16 active or none of a group), added in the order of the
// exchanges with lane ^ TPR / 2, ..., lane ^ 1, without the LDS crossbar: once lanes i and i ^ 8 hold the same sum, what
// stands four lanes back in the row of 16 is what stands at i ^ 4.
template <int CTRL>
MRL_DEV float dpp_add(float x) {
    return x + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xF, 0xF, true));
}
template <int TPR>
MRL_DEV float butterfly_sum(float x) {
    static_assert(TPR == 4 || TPR == 16, "a quad or a row of lanes");
    if constexpr (TPR == 16) x = dpp_add<0x128>(x);                       // row_ror:8
    if constexpr (TPR == 16) x = dpp_add<0x124>(x);                       // row_ror:4
    x = dpp_add<0x4E>(x);                                                 // quad_perm [2, 3, 0, 1]
    return dpp_add<0xB1>(x);                                              // quad_perm [1, 0, 3, 2]
}

// head_rows of mlp_tile.hpp for 16 rows; PITCH = floats per padded weight row in w2s (PA_MAX for a
// head staged with stage_head, 1 for a single-output head stored as a plain column followed by its
// bias).  Same lane split per row and same butterfly, hence the same bits as head_rows.  Serial latency bounds it (2.8 to 3.7
// thousand cycles of a rollout step, of 24 to 46): all of a lane's operands are requested ahead of its products, and the
// sums go over the lanes in DPP instructions instead of the LDS crossbar; CartPole, hidden width 64, 1024 envs 2.70 : 2.50
// us per step, LunarLander, hidden width 256, 4096 envs 19.3 : 18.7.
template <int H, int NA, int PITCH>
MRL_DEV void head_row16(const float *w2s, const float *h2, int r, int part, float (&out)[NA]) {
    constexpr int CP = 16, TPR = H / CP, BLK = NA == 8 ? 8 : 16;
    static_assert(64 % TPR == 0, "the lanes of a row sit in one wavefront");
    static_assert(NA == 1 || (PITCH == PA_MAX && (NA == 4 || NA == 8)), "one float, one float4 or two per padded row");
    const float *b2 = w2s + H * PITCH;
    float acc[NA];
#pragma unroll
    for (int a = 0; a < NA; ++a) acc[a] = 0.0f;
    // (element i is column (i + part) & 15 of the part: up to 15 - part it lies i behind the first, then 16 less)
    const float *hp = h2 + r * (H + 1) + part * CP + part, *wp = w2s + (part * CP + part) * PITCH;
#pragma unroll
    for (int b = 0; b < CP; b += BLK) {
        float hv[BLK], wv[BLK][NA];
#pragma unroll
        for (int j = 0; j < BLK; ++j) {
            const int i = b + j, back = i + part < CP ? 0 : CP;
            hv[j] = hp[i - back];
            const float *w = wp + (i - back) * PITCH;
            if (NA == 1) {
                wv[j][0] = w[0];
            } else {
#pragma unroll
                for (int a = 0; a < NA; a += 4) {
                    const float4 x = *reinterpret_cast<const float4 *>(w + a);
                    wv[j][a] = x.x; wv[j][a + 1] = x.y; wv[j][a + 2] = x.z; wv[j][a + 3] = x.w;
                }
            }
        }
#pragma unroll
        for (int j = 0; j < BLK; ++j) {
#pragma unroll
            for (int a = 0; a < NA; ++a) acc[a] = fmaf(hv[j], wv[j][a], acc[a]);
        }
    }
#pragma unroll
    for (int a = 0; a < NA; ++a) out[a] = butterfly_sum<TPR>(acc[a]) + b2[a];   // (in all lanes of the row)
}
// The same, of one or two outputs, with a lane's weights in registers from call to call.
template <int H, int NA, int PITCH>
struct HeadRow16 {
    static constexpr int CP = 16, TPR = H / CP;
    float w[CP][NA], b[NA];
    MRL_DEV void load(const float *w2s, int part) {
#pragma unroll
        for (int a = 0; a < NA; ++a) {
            b[a] = w2s[H * PITCH + a];
#pragma unroll
            for (int i = 0; i < CP; ++i) w[i][a] = w2s[(part * CP + ((i + part) & (CP - 1))) * PITCH + a];
        }
    }
    MRL_DEV void sums(const float *h2, int r, int part, float (&out)[NA]) const {
        const float *hp = h2 + r * (H + 1) + part * CP + part;
        float hv[CP], acc[NA];
#pragma unroll
        for (int i = 0; i < CP; ++i) hv[i] = hp[i - (i + part < CP ? 0 : CP)];
#pragma unroll
        for (int a = 0; a < NA; ++a) acc[a] = 0.0f;
#pragma unroll
        for (int i = 0; i < CP; ++i)
#pragma unroll
            for (int a = 0; a < NA; ++a) acc[a] = fmaf(hv[i], w[i][a], acc[a]);
#pragma unroll
        for (int a = 0; a < NA; ++a) out[a] = butterfly_sum<TPR>(acc[a]) + b[a];
    }
};
template <int H, int NA, int PITCH>
MRL_DEV void head_rows16(const float *w2s, int A, const float *h2, float *out, int out_ld, int t, int nthreads) {
    constexpr int TPR = H / 16;
    for (int pair = t; pair < PR16 * TPR; pair += nthreads) {
        const int r = pair / TPR, part = pair % TPR;
        float v[NA];
        head_row16<H, NA, PITCH>(w2s, h2, r, part, v);
#pragma unroll
        for (int a = 0; a < NA; ++a)
            if (part == 0 && a < A) out[r * out_ld + a] = v[a];
    }
}

template <int H>
MRL_DEV void head16(const float *w2s, int A, const float *h2, float *out, int out_ld, int t, int nthreads) {
    if constexpr (H == 128) head_chain<H, PR16, PA_MAX>(w2s, A, h2, out, out_ld, t);
    else if (A == 1) head_rows16<H, 1, PA_MAX>(w2s, A, h2, out, out_ld, t, nthreads);
    else if (A <= 4) head_rows16<H, 4, PA_MAX>(w2s, A, h2, out, out_ld, t, nthreads);
    else head_rows16<H, 8, PA_MAX>(w2s, A, h2, out, out_ld, t, nthreads);
}

// the critic's head: weights as a plain column of H, then the bias
template <int H>
MRL_DEV void head16_value(const float *w2c, const float *h2, float *out, int t, int nthreads) {
    if constexpr (H == 128) head_chain<H, PR16, 1>(w2c, 1, h2, out, 1, t);
    else head_rows16<H, 1, 1>(w2c, 1, h2, out, 1, t, nthreads);
}

}  // namespace mrl
