// gasp_cnn_stream.h -- the surrogate network for L <= 64, its layers joined in LDS
// instead of through memory.
//
// The layers one by one (gasp_cnn.hip, still the path for L >= 128) write and
// read 64 bytes a position and layer: 8.6 GB for 4096 grids of 64 x 64, 1.7 GB
// for a training batch of 256, and that traffic, not the matrix cores, set the
// time.  Here
//  - net_fwd carries an image from spins to pooled features in one pass (in
//    training it also stores a2, a3, a bit per channel of a4 and conv1's table
//    index, 2 bytes a position);
//  - net_back<k> (k = 4, 3, 2) reads dz_k and a_(k-1) once for both the weight
//    gradient and dz_(k-1); layer 4 makes dz_4 from the mask bits and the pooled
//    gradient, layer 2 makes a1 from the indices;
//  - net_reduce sums every layer's partial gradients and, in training, applies
//    Adam and writes the new weights' fragments.
// In training every sum is taken in the order of the separate kernels (a tap after
// the other, bands of four rows in chains, partials in chunks of 32), so activations,
// gradients and trained weights are theirs bit for bit.  Inference has the same
// activations, but pools them by eight rows (net_fwd): a grid's pB is the same bits
// whatever the batch (of +-1, see below), and differs from the separate kernels' by
// float32 rounding.
//
// The four 16-byte chunks of a position p (64 bytes) lie in LDS at chunk ^ ((p >>
// 2) & 3), which puts the fragment reads of 16 consecutive positions on 16
// different bank quads.
//
// L <= 64, as a ring row holds 64 columns: with 128 the two rings take 200 KB, more
// than a CU's LDS (strips of columns with halos, which would fit, were not tried).
//
// conv1 has one input channel of +-1, so a1 at a position is one of 512 rows,
// found by the nine spins around it: a table of 512 x 32 bfloat16 takes its
// place, and layer 2's fragments are read from the table.  A batch that holds any
// other value (net_fwd finds out, `odd`) is evaluated by the separate kernels
// instead: net_head then writes kNotSpins and net_reduce takes no step, and the
// host runs the batch again.
#pragma once

namespace cnn {

constexpr int kSP = 72;             // net_fwd: positions per ring row (64 columns, up to 8 halo columns)
constexpr int kSRow = kSP * 64;     // bytes per ring row
constexpr int kSBlk = 4 * kSRow;    // a block: four rows; a ring: three blocks
constexpr int kFwdTab = 0;          // conv1's table, then the rings of a2 and a3
constexpr int kFwdR2 = 512 * 64;
constexpr int kFwdR3 = kFwdR2 + 3 * kSBlk;
constexpr int kFwdCode = kFwdR3 + 3 * kSBlk;      // table offsets [2][6 rows][kSP], 2 bytes
constexpr int kFwdBits = kFwdCode + 2 * 6 * kSP * 2;  // spins [2 units][64 rows], 64 bits
constexpr int kFwdRow = kFwdBits + 2 * 64 * 8;  // tab_row of every code, 2 bytes
constexpr int kFwdLds = kFwdRow + 512 * 2;
// net_back: two windows (six rows of L + 2 positions) of dz_k and of a_(k-1), then
// the sums of half of the gradient waves
constexpr int back_win(int L) { return 6 * (L + 2) * 64; }
constexpr int kBackRed = 2 * 18 * 64 * 16;
constexpr int back_lds(int L) { return 4 * back_win(L) + kBackRed + 2 * 16 * 4; }
constexpr int kFwdThreads = 768, kBackThreads = 512, kRedThreads = 1024;

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
#define LDS_AS __attribute__((address_space(3)))
// These kernels declare no static LDS: LDS byte x is address x.
__device__ __forceinline__ u32x4 lds16(uint32_t a) { return *(const LDS_AS u32x4 *)(uintptr_t)a; }
__device__ __forceinline__ void lds16_set(uint32_t a, u32x4 v) { *(LDS_AS u32x4 *)(uintptr_t)a = v; }
__device__ __forceinline__ uint64_t lds8(uint32_t a) { return *(const LDS_AS uint64_t *)(uintptr_t)a; }
__device__ __forceinline__ uint32_t lds2(uint32_t a) { return *(const LDS_AS uint16_t *)(uintptr_t)a; }
__device__ __forceinline__ void lds2_set(uint32_t a, uint32_t v) { *(LDS_AS uint16_t *)(uintptr_t)a = (uint16_t)v; }
__device__ __forceinline__ LDS_AS float *ldsf(uint32_t a) { return (LDS_AS float *)(uintptr_t)a; }
// Four positions x 16 channels per 16 lanes, transposed: lane i names position
// i / 4, channels 4 (i % 4) and gets channel i of the four positions.
__device__ __forceinline__ u32x2 lds_tr(uint32_t a) {
    return __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((LDS_AS s16x4 *)(uintptr_t)a));
}
__device__ __forceinline__ uint32_t swz(int p, int chunk) {
    return (uint32_t)(p * 64 + 16 * (chunk ^ ((p >> 2) & 3)));
}
__device__ __forceinline__ f32x4 mfma4(u32x4 a, u32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
// two floats to bfloat16, to nearest even
__device__ __forceinline__ uint32_t bf_pack(float a, float b) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, bf16x2));
}
// A tile's D registers (channels 16 h + 4 kq + j of one position per lane, two
// halves packed as x, y) to eight consecutive channels a lane: chunk out_chunk(kq).
__device__ __forceinline__ u32x4 to_chunk(uint32_t x0, uint32_t y0, uint32_t x1, uint32_t y1) {
    const auto x = __builtin_amdgcn_permlane16_swap(x0, x1, false, false);
    const auto y = __builtin_amdgcn_permlane16_swap(y0, y1, false, false);
    return u32x4{x[0], y[0], x[1], y[1]};
}
__device__ __forceinline__ int out_chunk(int kq) { return ((kq & 1) << 1) | (kq >> 1); }

// net_fwd's units.  64 / L images lie side by side in 64 columns (a group); a unit
// is a band of Rb rows of a group, and a workgroup takes units blockIdx.x + k
// gridDim.x in turn as one stream of blocks of four rows, P to a unit.  A ring row
// holds a halo column on each side of every image.
struct Stream {
    int k = 0, j = 0;
    __device__ __forceinline__ void next(int P) {
        if (++j == P) {
            j = 0;
            ++k;
        }
    }
};
template <int V>
struct Role {
    static constexpr int value = V;
};
struct NetShape {
    int n, nb, Rb, units;  // images, bands per group, rows per band
    __device__ __forceinline__ int unit(int k) const { return (int)blockIdx.x + k * (int)gridDim.x; }
    __device__ __forceinline__ int group(int u) const { return u / nb; }
    __device__ __forceinline__ int first_row(int u) const { return (u % nb) * Rb; }
    // units of this workgroup
    __device__ __forceinline__ int count() const {
        return (int)blockIdx.x < units ? (units - 1 - (int)blockIdx.x) / (int)gridDim.x + 1 : 0;
    }
};

// Zero if the four bytes are all +1 or -1: bit 0 set, the others alike.
__device__ __forceinline__ uint32_t not_spins(uint32_t v) {
    return ((v ^ (v >> 1)) & 0x7E7E7E7Eu) | (~v & 0x01010101u);
}
constexpr uint32_t kNotSpins = 0x7FC51D05u;  // net_head's "pB" of a batch that is not +-1: a NaN

// Spins of a group as one 64-bit mask per row (bit = column, 1 = up) to LDS;
// absent images give zeros.  One thread per 16 columns: `it` < 4 L.  True if some
// value is not +-1.
template <int LG>
__device__ __forceinline__ bool load_bits(const int8_t *__restrict__ s, int n, int img0, uint32_t to, int it) {
    constexpr int L = 1 << LG;
    const int row = it >> 2, col = (it & 3) * 16, img = img0 + (col >> LG);
    uint32_t bits = 0u, bad = 0u;
    if (img < n) {
        const u32x4 v = *(const u32x4 *)(s + (size_t)img * (L * L) + row * L + (col & (L - 1)));
#pragma unroll
        for (int q = 0; q < 4; ++q) bits |= ((((~v[q] >> 7) & 0x01010101u) * 0x01020408u) >> 24 & 0xFu) << (4 * q);
        bad = not_spins(v[0]) | not_spins(v[1]) | not_spins(v[2]) | not_spins(v[3]);
    }
    lds2_set(to + 8u * (uint32_t)row + 2u * (uint32_t)(it & 3), bits);
    return bad != 0u;
}
// The nine spins around (row, col) as conv1's table index (bit t = tap t).
template <int LG>
__device__ __forceinline__ uint32_t code_at(uint32_t bits, int row, int col) {
    constexpr int L = 1 << LG;
    const int c = col & (L - 1), base = col - c;
    uint32_t code = 0u;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        const uint64_t m = lds8(bits + 8u * (uint32_t)((row + d - 1) & (L - 1)));
        const uint32_t lo = (uint32_t)m, hi = (uint32_t)(m >> 32);
        uint32_t w;
        if constexpr (LG == 6) {
            // columns col - 1 .. col + 1 of the ring of 64: a funnel shift
            const int r = (col - 1) & 63;
            w = __builtin_amdgcn_alignbit(r < 32 ? hi : lo, r < 32 ? lo : hi, (uint32_t)r);
        } else if constexpr (LG == 5) {
            const uint32_t x = col < 32 ? lo : hi;
            w = __builtin_amdgcn_alignbit(x, x, (uint32_t)(c - 1));
        } else {
            const uint32_t x = ((col < 32 ? lo : hi) >> (base & 16)) & 0xFFFFu;  // 16 columns, twice
            w = (x | (x << 16)) >> ((c - 1) & 15);
        }
        code |= (w & 7u) << (3 * d);
    }
    return code;
}

// LDS offset of conv1's table row for nine spins (its chunk q at offset ^ 16 q).
// Rows that grids often need at once, those of the empty neighbourhood and of
// one odd spin, must not share banks: each spin's bit toggles its own non-zero
// 4-bit pattern of (256-byte quarter of the banks, chunk).
__device__ __forceinline__ uint32_t tab_row(uint32_t nine) {
    constexpr uint32_t kHash[9] = {4, 8, 1, 2, 12, 3, 5, 10, 15};
    uint32_t h = 0u;
#pragma unroll
    for (int t = 0; t < 9; ++t) h ^= (nine >> t) & 1u ? kHash[t] : 0u;
    return ((nine & ~3u) | (h >> 2)) * 64u + 16u * (h & 3u);
}

// R rows x 16 positions x 32 output channels of a 3x3 convolution: frag(r, dx) is
// the B fragment of window row r (0 .. R + 1) shifted by dx - 1.  A fragment serves
// up to three output rows: with four rows 18 reads feed 72 MFMAs.  done(o, sums) is
// called as soon as row o has its last tap, so that its packing and stores run
// beside the next rows' MFMAs.
template <int R, class F, class D>
__device__ __forceinline__ void conv_block(const u32x4 (&wa)[9][2], F frag, D done) {
    f32x4 acc[R][2];
#pragma unroll
    for (int o = 0; o < R; ++o)
#pragma unroll
        for (int h = 0; h < 2; ++h) acc[o][h] = f32x4{0.f, 0.f, 0.f, 0.f};
    u32x4 f[2][3];
#pragma unroll
    for (int dx = 0; dx < 3; ++dx) f[0][dx] = frag(0, dx);
#pragma unroll
    for (int r = 0; r < R + 2; ++r) {
        if (r < R + 1) {
#pragma unroll
            for (int dx = 0; dx < 3; ++dx) f[(r + 1) & 1][dx] = frag(r + 1, dx);
        }
        __builtin_amdgcn_sched_barrier(0);  // the next row's reads go out before this row's MFMAs
#pragma unroll
        for (int dx = 0; dx < 3; ++dx)
#pragma unroll
            for (int o = 0; o < R; ++o) {
                const int dy = r - o;
                if (dy < 0 || dy > 2) continue;
#pragma unroll
                for (int h = 0; h < 2; ++h) acc[o][h] = mfma4(wa[3 * dy + dx][h], f[r & 1][dx], acc[o][h]);
            }
        if (r >= 3) done(r - 3, acc[r - 3]);
    }
    done(R - 1, acc[R - 1]);
}
// Sum over the 16 lanes of a row, the butterfly over lane ^ 1, 2, 4 and 8 (once the
// lanes of a quad agree, a mirrored half row gives what lane ^ 4 holds).
template <int CTRL>
__device__ __forceinline__ float dpp_move(float v) {
    return __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(v), CTRL, 0xf, 0xf, true));
}
__device__ __forceinline__ float sum16(float v) {
    v += dpp_move<0xB1>(v);    // quad_perm [1, 0, 3, 2]
    v += dpp_move<0x4E>(v);    // quad_perm [2, 3, 0, 1]
    v += dpp_move<0x141>(v);   // row_half_mirror
    return v + dpp_move<0x140>(v);  // row_mirror
}
// OR of a value over the four lanes of a position (lane, lane ^ 16, ^ 32, ^ 48)
__device__ __forceinline__ uint32_t or_quarters(uint32_t m) {
    const auto x = __builtin_amdgcn_permlane16_swap(m, m, false, false);
    m = x[0] | x[1];
    const auto y = __builtin_amdgcn_permlane32_swap(m, m, false, false);
    return y[0] | y[1];
}

// ------------------------------------------------------------------ forward
// Twelve waves, four per layer 2, 3 and 4, each on its 16 columns: in a step
// (one barrier) a layer's waves compute a block of four rows while the next
// layer works two blocks behind, so each ring holds three blocks.  Block j of a
// unit is a2's rows 4j - 2 .. 4j + 1, a3's 4j - 1 .. 4j + 2 and a4's 4j .. 4j + 3
// of the band (a band takes Rb / 4 + 1 blocks: two rows of a2 and one of a3 are
// computed again above and below it).
// What bounds it (4096 grids of L = 64): the matrix cores are busy 57 to 65% of
// the cycles (at the 1.95 GHz that the card then runs), the rest is the waves'
// packing and stores between barriers; LDS is busy half of the time.  727 us
// against 372 + 3 x 663 + 198 for the layers one by one.  The first form took 834:
// conv2's waves made the table offsets themselves, rows of the table that grids
// need together shared banks, and a step's reads went out as they were needed.
// pool, training: [unit][wave][set][32], sums of a4 over a wave's 16 columns and
// the unit's rows, those of each residue mod 64 / L apart (as `head` adds them).
// pool, inference: [group][eight rows][wave][32], so that an image's sums do not
// depend on the bands that the number of images leads to (with a sum per unit a
// grid's pB moved in its last bits with the size of the batch).  Written 16 bytes a
// lane that costs nothing: 1024 grids of L = 64 180 us, 181 with a sum per unit,
// 185 written 4 bytes a lane.
// a4: only where bands leave the pooling to `head` (else NULL).
// m4[image][position]: bit c set where a4 > 0.  tab, code: conv1's table and every
// position's index in it, for net_back<2>.
template <bool TRAIN, int LG>
__global__ void __launch_bounds__(kFwdThreads) net_fwd(const int8_t *__restrict__ s, const uint16_t *__restrict__ wf,
                                                       const float *__restrict__ p, const float *__restrict__ w1r,
                                                       uint16_t *__restrict__ a2, uint16_t *__restrict__ a3,
                                                       uint16_t *__restrict__ a4, uint32_t *__restrict__ m4,
                                                       float *__restrict__ pool, uint16_t *__restrict__ tab,
                                                       uint16_t *__restrict__ code, int *__restrict__ odd, NetShape g) {
    constexpr int L = 1 << LG, N = L * L, kSets = 64 >> LG;  // kSets images in a group
    constexpr int kAcc = TRAIN ? kSets : 1;
    const int tid = threadIdx.x, lane = tid & 63, w4 = (tid >> 6) & 3;
    const int role = __builtin_amdgcn_readfirstlane(tid >> 8);  // 0, 1, 2: conv2, conv3, conv4
    const int K = g.count(), P = g.Rb / 4 + 1;
    {
        const int c2 = tid & 15;  // channels 2 c2 and 2 c2 + 1 of rows tid / 16 + 48 k
        float w[2][10];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            w[h][9] = p[OFF_B1 + 2 * c2 + h];
#pragma unroll
            for (int t = 0; t < 9; ++t) w[h][t] = w1r[t * C + 2 * c2 + h];
        }
        for (int nine = tid >> 4; nine < 512; nine += kFwdThreads / 16) {
            uint32_t out = 0u;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                float z = w[h][9];
#pragma unroll
                for (int t = 0; t < 9; ++t) z += w[h][t] * (((nine >> t) & 1) ? 1.0f : -1.0f);
                out |= (uint32_t)f2bf(fmaxf(z, 0.0f)) << (16 * h);
            }
            const uint32_t row = tab_row((uint32_t)nine);
            *(LDS_AS uint32_t *)(uintptr_t)(kFwdTab + (row ^ (16u * (uint32_t)(c2 >> 2))) + 4u * (uint32_t)(c2 & 3)) = out;
            if (c2 == 0) lds2_set(kFwdRow + 2u * (uint32_t)nine, row);
            if (TRAIN && blockIdx.x == 0) ((uint32_t *)tab)[nine * 16 + c2] = out;
        }
    }
    if (tid < 4 * L && load_bits<LG>(s, g.n, g.group(g.unit(0)) * kSets, kFwdBits, tid)) *odd = 1;
    __syncthreads();
    // table offsets of a2 block j's six a1 rows, 4j - 3 .. 4j + 2
    auto codes = [&](const Stream &st, int buf) {
        const uint32_t bits = kFwdBits + (uint32_t)(st.k & 1) * 512u;
        const int u = g.unit(st.k), y0 = g.first_row(u), yr = 4 * st.j - 3;
        for (int e = tid & 255; e < 6 * 64; e += 256) {
            const int q = e >> 6, col = e & 63;
            const uint32_t nine = code_at<LG>(bits, (y0 + yr + q) & (L - 1), col);
            const uint32_t off = lds2(kFwdRow + 2u * nine);
            const uint32_t row = kFwdCode + (uint32_t)(buf * 6 + q) * (kSP * 2);
            const int c = col & (L - 1), first = (col >> LG) * (L + 2);
            if (TRAIN) {  // rows 4j - 2 .. 4j + 1, each once
                const int img = g.group(u) * kSets + (col >> LG);
                if (q >= 1 && q <= 4 && yr + q >= 0 && yr + q < g.Rb && img < g.n)
                    code[(size_t)img * N + (size_t)(y0 + yr + q) * L + c] = (uint16_t)nine;
            }
            lds2_set(row + 2u * (uint32_t)(first + 1 + c), off);
            if (c == 0) lds2_set(row + 2u * (uint32_t)(first + L + 1), off);
            if (c == L - 1) lds2_set(row + 2u * (uint32_t)first, off);
        }
    };
    if (role == 0) codes(Stream{}, 0);
    __syncthreads();

    const int pl = lane & 15, kq = lane >> 4;
    const int im = (16 * w4) >> LG, c = ((16 * w4) & (L - 1)) + pl;
    const int first = im * (L + 2);  // position of the image's left halo column
    uint32_t off[3];
#pragma unroll
    for (int dx = 0; dx < 3; ++dx) off[dx] = swz(first + c + dx, kq);
    const int oc = out_chunk(kq);
    const uint32_t oof = swz(first + 1 + c, oc);
    const int hp = c == 0 ? first + L + 1 : first;  // the other side's halo position, for the outer columns
    const bool halo = c == 0 || c == L - 1;
    const uint32_t hof = swz(hp, oc);
    // a loop (and registers) for each layer's waves, with the same barriers
    auto run = [&](auto role_of) {
        constexpr int layer = decltype(role_of)::value;
        u32x4 wa[9][2];
#pragma unroll
        for (int t = 0; t < 9; ++t)
#pragma unroll
            for (int h = 0; h < 2; ++h) wa[t][h] = ((const u32x4 *)wf)[((layer * 9 + t) * 2 + h) * 64 + lane];
        const float *bp = p + OFF_B[2 + layer];
        float bias[2][4];
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int j = 0; j < 4; ++j) bias[h][j] = bp[16 * h + 4 * kq + j];
        float psum[kAcc][8];
#pragma unroll
        for (int q = 0; q < kAcc; ++q)
#pragma unroll
            for (int e = 0; e < 8; ++e) psum[q][e] = 0.f;

        Stream st;  // the layer's own block
        const int lag = 2 * layer, total = K * P;
        int slot = 0;  // of block st in the layer's input ring (layers 3, 4) and in its output ring
        Stream cs;  // layer 3's waves, the least busy: conv2's block of this step
        uint64_t bad = 0u;  // lanes that met other values than +-1 (a scalar: no vector register is left)
        for (int step = 0; step < total + 4; ++step) {
            const int i = step - lag;
            if (layer == 1 && step < total) {
                // the next unit's spins, then the next block's table offsets
                if (cs.j == 0 && cs.k + 1 < K) {
                    bool here = false;
                    if ((tid & 255) < 4 * L)
                        here = load_bits<LG>(s, g.n, g.group(g.unit(cs.k + 1)) * kSets, kFwdBits + (uint32_t)((cs.k + 1) & 1) * 512u, tid & 255);
                    bad |= __builtin_amdgcn_ballot_w64(here);
                }
                cs.next(P);
                if (step + 1 < total) codes(cs, (step + 1) & 1);
            }
            if (i >= 0 && i < total) {
                const int slot1 = slot == 2 ? 0 : slot + 1;
                const int u = g.unit(st.k), img = g.group(u) * kSets + im, y0 = g.first_row(u);
                const int yb = 4 * st.j - 2 + layer;  // the block's first row in the band
                uint32_t x[2], y[2];
                auto pack = [&](f32x4 (&d)[2]) {
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        x[h] = bf_pack(fmaxf(d[h][0] + bias[h][0], 0.f), fmaxf(d[h][1] + bias[h][1], 0.f));
                        y[h] = bf_pack(fmaxf(d[h][2] + bias[h][2], 0.f), fmaxf(d[h][3] + bias[h][3], 0.f));
                    }
                };
                // layers 2 and 3: row o to the next layer's ring, and in training to memory
                const uint32_t to = (layer == 0 ? kFwdR2 : kFwdR3) + (uint32_t)slot * kSBlk;
                uint16_t *keep = layer == 0 ? a2 : a3;
                auto row_out = [&](int o, f32x4 (&d)[2]) {
                    pack(d);
                    const u32x4 v = to_chunk(x[0], y[0], x[1], y[1]);
                    lds16_set(to + (uint32_t)(o * kSRow) + oof, v);
                    if (halo) lds16_set(to + (uint32_t)(o * kSRow) + hof, v);
                    const int row = yb + o;
                    if (TRAIN && row >= 0 && row < g.Rb && img < g.n)
                        *(u32x4 *)(keep + ((size_t)img * N + (size_t)(y0 + row) * L + c) * C + 8 * oc) = v;
                };
                auto ring_frag = [&](uint32_t ring) {
                    const uint32_t A = ring + (uint32_t)slot * kSBlk, B = ring + (uint32_t)slot1 * kSBlk;
                    return [=, &off](int r, int dx) {
                        return lds16((r < 4 ? A + (uint32_t)(r * kSRow) : B + (uint32_t)((r - 4) * kSRow)) + off[dx]);
                    };
                };
                if constexpr (layer == 0) {
                    const uint32_t cb = kFwdCode + (uint32_t)(i & 1) * (6 * kSP * 2) + 2u * (uint32_t)(first + c);
                    const uint32_t q16 = 16u * (uint32_t)kq;
                    conv_block<4>(
                        wa,
                        [&](int r, int dx) { return lds16(kFwdTab + (lds2(cb + (uint32_t)(r * kSP * 2 + 2 * dx)) ^ q16)); },
                        row_out);
                } else if constexpr (layer == 1) {
                    conv_block<4>(wa, ring_frag(kFwdR2), row_out);
                } else if (st.j < P - 1) {
                    conv_block<4>(wa, ring_frag(kFwdR3), [&](int o, f32x4 (&d)[2]) {
                        pack(d);
                        float(&ps)[8] = psum[o % kAcc];
#pragma unroll
                        for (int h = 0; h < 2; ++h) {
                            ps[4 * h] += __uint_as_float(x[h] << 16);
                            ps[4 * h + 1] += __uint_as_float(x[h] & 0xFFFF0000u);
                            ps[4 * h + 2] += __uint_as_float(y[h] << 16);
                            ps[4 * h + 3] += __uint_as_float(y[h] & 0xFFFF0000u);
                        }
                        if (TRAIN) {
                            uint32_t m = 0u;
#pragma unroll
                            for (int h = 0; h < 2; ++h) {
                                m |= ((x[h] & 0xFFFFu) ? 1u : 0u) << (16 * h);
                                m |= ((x[h] >> 16) ? 2u : 0u) << (16 * h);
                                m |= ((y[h] & 0xFFFFu) ? 4u : 0u) << (16 * h);
                                m |= ((y[h] >> 16) ? 8u : 0u) << (16 * h);
                            }
                            m = or_quarters(m << (4 * kq));
                            const size_t pos = (size_t)img * N + (size_t)(y0 + yb + o) * L + c;
                            if (kq == 0 && img < g.n) m4[pos] = m;
                            if (a4 && img < g.n) *(u32x4 *)(a4 + pos * C + 8 * oc) = to_chunk(x[0], y[0], x[1], y[1]);
                        }
                    });
                    // training: the unit's last block; inference: every eight rows
                    if (TRAIN ? st.j == P - 2 : (st.j & 1) != 0) {
                        const size_t to = TRAIN ? (size_t)u : (size_t)g.group(u) * (L / 8) + (size_t)(y0 + 4 * st.j) / 8;
                        f32x4 *out = (f32x4 *)(pool + (to * 4 + w4) * kAcc * C + 4 * kq);
#pragma unroll
                        for (int q = 0; q < 2 * kAcc; ++q) {
                            f32x4 v;
#pragma unroll
                            for (int j = 0; j < 4; ++j) {
                                v[j] = sum16(psum[q / 2][4 * (q & 1) + j]);
                                psum[q / 2][4 * (q & 1) + j] = 0.f;
                            }
                            if (pl == 0) out[4 * q] = v;
                        }
                    }
                }
                st.next(P);
                slot = slot1;
            }
            __syncthreads();
        }
        if (layer == 1 && bad) *odd = 1;
    };
    if (role == 0) run(Role<0>{});
    else if (role == 1) run(Role<1>{});
    else run(Role<2>{});
}

// The head of one image per wave: pooled features from net_fwd's sums, then as
// `head` (gasp_cnn.hip).
template <bool TRAIN, int LG>
__global__ void __launch_bounds__(64) net_head(const float *__restrict__ pool, const float *__restrict__ p,
                                               const float *__restrict__ labels, float *__restrict__ pb,
                                               float *__restrict__ loss, float *__restrict__ part_head,
                                               float *__restrict__ dg, const int *__restrict__ odd, NetShape g,
                                               float inv_batch) {
    __shared__ float gs[C], dh[HID];
    const int img = blockIdx.x, t = threadIdx.x;
    const bool refuse = !TRAIN && *odd != 0;
    constexpr int L = 1 << LG, kSets = 64 >> LG, kAcc = TRAIN ? kSets : 1, kStrips = L / 16;
    const int group = img / kSets, im = img % kSets;
    if (t < C) {
        float v = 0.f;
        const int parts = TRAIN ? g.nb : L / 8;
        for (int b = 0; b < parts; ++b)
            for (int q = 0; q < kAcc; ++q)
                for (int w = 0; w < kStrips; ++w)
                    v += pool[(((size_t)group * parts + b) * 4 + im * kStrips + w) * kAcc * C + q * C + t];
        gs[t] = v / (float)(L * L);
    }
    __syncthreads();
    float pre = p[OFF_FB1 + t];
#pragma unroll
    for (int k = 0; k < C; ++k) pre += gs[k] * p[OFF_FW1 + k * HID + t];
    const float h = fmaxf(pre, 0.f), w2 = p[OFF_FW2 + t];
    float z = h * w2;
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) z += __shfl_xor(z, off, 64);
    // one lane's sum for all: the first product may be fused into the first
    // addition, and then lanes 32 .. 63 round another way
    z = __uint_as_float((uint32_t)__builtin_amdgcn_readfirstlane((int)__float_as_uint(z))) + p[OFF_FB2];
    const float sig = 1.0f / (1.0f + expf(-z));
    if (t == 0) pb[img] = refuse ? __uint_as_float(kNotSpins) : sig;
    if (!TRAIN) return;
    const float y = labels[img];
    if (t == 0) loss[img] = fmaxf(z, 0.f) + log1pf(expf(-fabsf(z))) - y * z;
    const float dz = (sig - y) * inv_batch;
    float *ph = part_head + (size_t)img * HEAD_N;
    const float d = pre > 0.f ? dz * w2 : 0.f;
    ph[OFF_FW2 - OFF_FW1 + t] = h * dz;
    ph[OFF_FB1 - OFF_FW1 + t] = d;
    if (t == 0) ph[OFF_FB2 - OFF_FW1] = dz;
    dh[t] = d;
#pragma unroll 8
    for (int k = 0; k < C; ++k) ph[k * HID + t] = gs[k] * d;
    __syncthreads();
    if (t < C) {
        float v = 0.f;
        for (int j = 0; j < HID; ++j) v += dh[j] * p[OFF_FW1 + t * HID + j];
        dg[img * C + t] = v;
    }
}

// ------------------------------------------------------------------ backward
// Layer KL = 4, 3, 2.  A band is four rows of an image; chain b of the weight
// gradient is the bands b, b + chains, b + 2 chains, ..., whose sum is one row of
// part, [9][ci][co] and the bias (conv_wgrad's workgroups).  A workgroup takes
// chains in turn, band after band: in a step all threads load the next band's
// windows (rows y0 - 1 .. y0 + 4 of dz_k and a_(k-1)) to registers, compute with
// the present ones in LDS, and store.  Eight waves:
//  - waves 0 .. 3 compute dz_(k-1) (conv_block with the transposed, tap-flipped
//    weights, masked by a_(k-1) > 0), 16 columns and L / 16 rows each;
//  - waves 4 .. 7 the weight gradient D[co][ci] += dz^T a: wave pair gc takes
//    every second run of 32 positions, wave nh of a pair one half of the input
//    channels.  Both operands are read transposed (ds_read_b64_tr_b16); at L = 64 a
//    band is 52 reads for 72 MFMAs.
// What bounds it: memory.  A layer at L = 64 with 256 images reads two tensors of
// 67 MB, writes one and 28 MB of partial rows in 57 us (4.0 TB/s; a large copy
// reaches 5.1 on this card); the matrix cores are busy a third of the time.
// conv_wgrad and conv_mfma took 46 + 47 us and read dz_k twice; head_bwd_fill, 42
// us, has no counterpart (layer 4 makes dz_4 here).
// At a chain's end pair 0 leaves its sums in LDS, and pair 1 adds its own to them
// and writes the row.  Workgroups of one XCD (blockIdx.x mod 8) run neighbouring
// chains, whose windows overlap, so that L2 serves the shared rows.
template <int KL, int LG>
__global__ void __launch_bounds__(kBackThreads) net_back(const uint16_t *__restrict__ dz, const uint32_t *__restrict__ m4,
                                                         const float *__restrict__ dg, const uint16_t *__restrict__ a,
                                                         const uint16_t *__restrict__ code, const uint16_t *__restrict__ wb,
                                                         uint16_t *__restrict__ out, float *__restrict__ part, int bands,
                                                         int chains) {
    constexpr int L = 1 << LG, N = L * L, kRowB = (L + 2) * 64, kWin = 6 * kRowB;
    constexpr uint32_t kZ = 0, kA = 2 * kWin, kRed = 4 * kWin, kRedB = kRed + kBackRed;
    constexpr int kItems = 6 * L * 4, kIt = (kItems + kBackThreads - 1) / kBackThreads;  // 16-byte items per window, per thread
    const int tid = threadIdx.x, lane = tid & 63, w4 = (tid >> 6) & 3;
    const bool data = __builtin_amdgcn_readfirstlane(tid >> 8) == 0;  // waves 0 .. 3
    const int pl = lane & 15, kq = lane >> 4;
    // chain t of this workgroup; chains in eight runs, one per XCD, where they divide
    const int G = (int)gridDim.x;
    const bool runs = (chains & 7) == 0 && (G & 7) == 0;
    auto chain = [&](int t) {
        const int b = (int)blockIdx.x;
        if (!runs) return b + t * G < chains ? b + t * G : -1;
        const int i = (b >> 3) + t * (G >> 3);
        return i < (chains >> 3) ? (b & 7) * (chains >> 3) + i : -1;
    };
    struct Walk {  // through the bands of this workgroup's chains
        int t, first, band;  // band < 0: done
    };
    auto after = [&](Walk w) {
        w.band += chains;
        if (w.band >= bands) {
            ++w.t;
            w.first = w.band = chain(w.t);
        }
        return w;
    };

    // loader: item tid + 512 q of a window is (row, column, chunk)
    const int lch = tid & 3;
    u32x4 vz[kIt], va[kIt];
    uint32_t nine[kIt];  // KL = 2: the table indices of the band after
    auto pos_of = [&](int band, int q, size_t *pos) {
        const int e = tid + kBackThreads * q, rr = e / (4 * L), col = (e % (4 * L)) >> 2;
        const int img = band / (L / 4), y = (4 * (band % (L / 4)) - 1 + rr) & (L - 1);
        *pos = (size_t)img * N + (size_t)(y * L + col);
        return kItems % kBackThreads == 0 || e < kItems;
    };
    auto load_codes = [&](int band) {
        if (KL != 2 || band < 0) return;
#pragma unroll
        for (int q = 0; q < kIt; ++q) {
            size_t pos;
            if (pos_of(band, q, &pos)) nine[q] = code[pos];
        }
    };
    auto load = [&](int band) {
        u32x4 dgv{};
        if constexpr (KL == 4) {
            const float inv = 1.0f / (float)N;
            const float *d = dg + (size_t)(band / (L / 4)) * C + 8 * lch;
#pragma unroll
            for (int q = 0; q < 4; ++q) dgv[q] = bf_pack(d[2 * q] * inv, d[2 * q + 1] * inv);
        }
#pragma unroll
        for (int q = 0; q < kIt; ++q) {
            size_t pos;
            if (!pos_of(band, q, &pos)) continue;
            if constexpr (KL == 4) {
                const uint32_t m = m4[pos] >> (8 * lch);
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    vz[q][e] = dgv[e] & (((m >> (2 * e)) & 1u ? 0xFFFFu : 0u) | ((m >> (2 * e)) & 2u ? 0xFFFF0000u : 0u));
            } else {
                vz[q] = *(const u32x4 *)(dz + pos * C + 8 * lch);
            }
            if constexpr (KL == 2) va[q] = *(const u32x4 *)(a + nine[q] * C + 8 * lch);  // a: conv1's table
            else va[q] = *(const u32x4 *)(a + pos * C + 8 * lch);
        }
    };
    auto store = [&](int buf) {
#pragma unroll
        for (int q = 0; q < kIt; ++q) {
            const int e = tid + kBackThreads * q, rr = e / (4 * L), col = (e % (4 * L)) >> 2;
            if (kItems % kBackThreads != 0 && e >= kItems) continue;
            const uint32_t row = (uint32_t)(buf * kWin + rr * kRowB), of = row + swz(1 + col, lch);
            lds16_set(kZ + of, vz[q]);
            lds16_set(kA + of, va[q]);
            if (col == 0 || col == L - 1) {
                const uint32_t ho = row + swz(col == 0 ? L + 1 : 0, lch);
                lds16_set(kZ + ho, vz[q]);
                lds16_set(kA + ho, va[q]);
            }
        }
    };
    Walk now{0, chain(0), chain(0)};  // grid <= chains: every workgroup has one
    Walk nxt = after(now);
    load_codes(now.band);
    load(now.band);
    store(0);
    load_codes(nxt.band);
    __syncthreads();

    // the steps; the two roles have loops (and registers) of their own, with the
    // same barriers: data waves hold 72 registers of weights and 32 of sums,
    // gradient waves 76 of sums and 32 of dz fragments
    auto steps = [&](auto compute, auto finish) {
        int ended = -1;  // the chain that ended in the step before
        for (int buf = 0; now.band >= 0; buf ^= 1) {
            if (nxt.band >= 0) load(nxt.band);
            if (ended >= 0) {
                finish(ended, true);
                __syncthreads();  // before the sums in LDS are written again
            }
            compute(kZ + (uint32_t)(buf * kWin), kA + (uint32_t)(buf * kWin));
            ended = nxt.t != now.t ? now.first : -1;
            if (ended >= 0) finish(ended, false);
            if (nxt.band >= 0) store(buf ^ 1);
            now = nxt;
            if (nxt.band >= 0) nxt = after(nxt);
            load_codes(nxt.band);
            __syncthreads();
        }
        finish(ended, true);
    };
    if (data) {
        constexpr int kStrips = L / 16, R = L / 16;
        u32x4 wa[9][2];
#pragma unroll
        for (int t = 0; t < 9; ++t)
#pragma unroll
            for (int h = 0; h < 2; ++h) wa[t][h] = ((const u32x4 *)wb)[(t * 2 + h) * 64 + lane];
        const int c = 16 * (w4 % kStrips) + pl, r0 = R * (w4 / kStrips);
        const int oc = out_chunk(kq);
        uint32_t off[3];
#pragma unroll
        for (int dx = 0; dx < 3; ++dx) off[dx] = (uint32_t)(r0 * kRowB) + swz(c + dx, kq);
        const uint32_t mof = (uint32_t)((r0 + 1) * kRowB) + swz(1 + c, oc);
        steps(
            [&](uint32_t z, uint32_t aw) {
                uint16_t *to = out + ((size_t)(now.band / (L / 4)) * N + (size_t)((4 * (now.band % (L / 4)) + r0) * L + c)) * C + 8 * oc;
                conv_block<R>(
                    wa, [&](int r, int dx) { return lds16(z + (uint32_t)(r * kRowB) + off[dx]); },
                    [&](int o, f32x4 (&d)[2]) {
                        u32x4 v = to_chunk(bf_pack(d[0][0], d[0][1]), bf_pack(d[0][2], d[0][3]), bf_pack(d[1][0], d[1][1]),
                                           bf_pack(d[1][2], d[1][3]));
                        const u32x4 m = lds16(aw + (uint32_t)(o * kRowB) + mof);
#pragma unroll
                        for (int q = 0; q < 4; ++q)
                            v[q] &= ((m[q] & 0xFFFFu) ? 0xFFFFu : 0u) | ((m[q] >> 16) ? 0xFFFF0000u : 0u);
                        *(u32x4 *)(to + o * L * C) = v;
                    });
            },
            [](int, bool) {});
    } else {
        constexpr int NK = L / 16;                            // runs of 32 positions of a pair per band
        constexpr int RS = LG == 6 ? 1 : 2;                   // rows from one to the next
        f32x4 acc[9][2];
        float bsum = 0.f;
#pragma unroll
        for (int t = 0; t < 9; ++t)
#pragma unroll
            for (int h = 0; h < 2; ++h) acc[t][h] = f32x4{0.f, 0.f, 0.f, 0.f};
        // run gc + 2 i: positions 32 (gc + 2 i) .. of the band's rows, 8 kq .. by this
        // lane; the lane names positions + pl / 4 and + 4 of them, channels 4 (pl % 4)
        const int gc = w4 >> 1, nh = w4 & 1;
        const int row0 = LG == 6 ? 0 : LG == 5 ? gc : 2 * gc + (kq >> 1);
        const int x0 = LG == 6 ? 32 * gc + 8 * kq : LG == 5 ? 8 * kq : 8 * (kq & 1);
        uint32_t zo[2][2], ao[3][2];
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const int x = x0 + 4 * q + (pl >> 2);
            auto of = [&](int half, int dx) {  // dx - 1: the tap's shift
                return swz(x + dx, 2 * half + ((pl & 3) >> 1)) + 8u * (uint32_t)(pl & 1);
            };
#pragma unroll
            for (int h = 0; h < 2; ++h) zo[h][q] = (uint32_t)((row0 + 1) * kRowB) + of(h, 1);
#pragma unroll
            for (int dx = 0; dx < 3; ++dx) ao[dx][q] = (uint32_t)(row0 * kRowB) + of(nh, dx);
        }
        steps(
            [&](uint32_t z, uint32_t aw) {
                u32x4 Z[NK][2];
#pragma unroll
                for (int i = 0; i < NK; ++i)
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        const uint32_t r = z + (uint32_t)(RS * i * kRowB);
                        const u32x2 lo = lds_tr(r + zo[h][0]), hi = lds_tr(r + zo[h][1]);
                        Z[i][h] = u32x4{lo[0], lo[1], hi[0], hi[1]};
                    }
                // the bias of channel half nh, as conv_wgrad adds it
#pragma unroll
                for (int i = 0; i < NK; ++i)
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const uint32_t v = nh ? Z[i][1][q] : Z[i][0][q];
                        bsum += __uint_as_float(v << 16) + __uint_as_float(v & 0xFFFF0000u);
                    }
#pragma unroll
                for (int r = 0; r < RS * (NK - 1) + 3; ++r)
#pragma unroll
                    for (int dx = 0; dx < 3; ++dx) {
                        const uint32_t row = aw + (uint32_t)(r * kRowB);
                        const u32x2 lo = lds_tr(row + ao[dx][0]), hi = lds_tr(row + ao[dx][1]);
                        const u32x4 b = {lo[0], lo[1], hi[0], hi[1]};
#pragma unroll
                        for (int i = 0; i < NK; ++i) {
                            const int dy = r - RS * i;
                            if (dy < 0 || dy > 2) continue;
#pragma unroll
                            for (int h = 0; h < 2; ++h) acc[3 * dy + dx][h] = mfma4(Z[i][h], b, acc[3 * dy + dx][h]);
                        }
                    }
            },
            [&](int ch, bool add) {
                if (add != (gc == 1)) return;
                bsum += __shfl_xor(bsum, 16, 64);
                bsum += __shfl_xor(bsum, 32, 64);  // lanes pl: channel 16 nh + pl
                float *row = part + (size_t)ch * kWgRow;
#pragma unroll
                for (int t = 0; t < 9; ++t)
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        LDS_AS f32x4 *d = (LDS_AS f32x4 *)(uintptr_t)(kRed + (uint32_t)(((nh * 9 + t) * 2 + h) * 64 + lane) * 16u);
                        if (add) *(f32x4 *)(row + t * C * C + (16 * nh + pl) * C + 16 * h + 4 * kq) = *d + acc[t][h];
                        else *d = acc[t][h];
                        acc[t][h] = f32x4{0.f, 0.f, 0.f, 0.f};
                    }
                if (kq == 0) {
                    LDS_AS float *d = ldsf(kRedB) + nh * 16 + pl;
                    if (add) row[9 * C * C + 16 * nh + pl] = *d + bsum;
                    else *d = bsum;
                }
                bsum = 0.f;
            });
    }
}

// ------------------------------------------------------------------ reduction
// g[j] = the sum of every partial row's entry j in reduce_chunks' order: chunks of
// kRedChunk rows each on its own, then the chunks' sums one after the other.  A
// workgroup takes 64 columns, sixteen chunks at a time.  With ADAM the parameters
// take their step and the new weights go to the fragment layouts (prep_weights).
struct NetParts {
    const float *part[5];  // conv1, conv2, conv3, conv4, head
    int rows[5];
};
struct AdamArgs {
    float lr, b1, b2, eps, c1, c2;
    const int *odd;  // no step if set (NULL: the data are known to be +-1)
};

template <bool ADAM>
__global__ void __launch_bounds__(kRedThreads) net_reduce(NetParts q, float *__restrict__ gout, float *__restrict__ p,
                                                          float *__restrict__ m, float *__restrict__ v,
                                                          uint16_t *__restrict__ wf, uint16_t *__restrict__ wb,
                                                          float *__restrict__ w1r, AdamArgs ad) {
    __shared__ float sums[16][64];
    constexpr int kCols[5] = {320, kWgRow, kWgRow, kWgRow, HEAD_N};
    constexpr int kDst[5] = {0, OFF_W[2], OFF_W[3], OFF_W[4], OFF_FW1};
    int blk = blockIdx.x, src = 0, ncol = 0, dst = 0;
    bool found = false;
#pragma unroll
    for (int i = 0; i < 5; ++i) {
        const int nblk = (kCols[i] + 63) / 64;
        if (!found && blk < nblk) {
            src = i;
            ncol = kCols[i];
            dst = kDst[i];
            found = true;
        }
        if (!found) blk -= nblk;
    }
    const int t = threadIdx.x & 63, rg = threadIdx.x >> 6, col = 64 * blk + t;
    const float *f = q.part[src] + (col < ncol ? col : 0);
    const int rows = q.rows[src], nc = (rows + kRedChunk - 1) / kRedChunk;
    float acc = 0.f;
    for (int c0 = 0; c0 < nc; c0 += 16) {
        const int r0 = (c0 + rg) * kRedChunk, r1 = min(rows, r0 + kRedChunk);
        float sum = 0.f;
#pragma unroll 8
        for (int r = r0; r < r1; ++r) sum += f[(size_t)r * ncol];
        sums[rg][t] = sum;
        __syncthreads();
        if (rg == 0)
            for (int i = 0; i < min(16, nc - c0); ++i) acc += sums[i][t];
        __syncthreads();
    }
    if (rg != 0 || col >= ncol) return;
    const int j = dst + col;
    gout[j] = acc;
    if constexpr (ADAM) {
        if (ad.odd && *ad.odd) return;
        const float gi = acc;
        const float mi = ad.b1 * m[j] + (1.f - ad.b1) * gi;
        const float vi = ad.b2 * v[j] + (1.f - ad.b2) * gi * gi;
        m[j] = mi;
        v[j] = vi;
        float w = p[j];
        w -= ad.lr * (mi / ad.c1) / (sqrtf(vi / ad.c2) + ad.eps);
        p[j] = w;
        if (src == 0) {
            if (col < 288) w1r[col] = bf2f(f2bf(w));
        } else if (src < 4 && col < 9 * C * C) {
            const int tap = col / (C * C), ci = (col / C) % C, co = col % C, k = src - 1;
            const uint16_t b = f2bf(w);
            wf[(((k * 9 + tap) * 2 + (co >> 4)) * 64 + ((co & 15) | ((ci >> 3) << 4))) * 8 + (ci & 7)] = b;
            wb[(((k * 9 + 8 - tap) * 2 + (ci >> 4)) * 64 + ((ci & 15) | ((co >> 3) << 4))) * 8 + (co & 7)] = b;
        }
    }
}
constexpr int kRedBlocks = 5 + 3 * ((kWgRow + 63) / 64) + (HEAD_N + 63) / 64;

}  // namespace cnn
