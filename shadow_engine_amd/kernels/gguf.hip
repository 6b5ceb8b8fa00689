// GGUF (Q8_0, IQ3_S) products y_j = W x_j for 1..8 inputs on the matrix cores (matvec_cols_*).
//
// Both formats' weights are a scale times small integers (Q8_0: codes of 8 bits, a scale a 32-block; IQ3_S: grid value * sign *
// (1 + 2 s), at most 465, one scale a 256-block), which f16 holds exactly.  A row of W is a column of operand B of
// v_mfma_f32_16x16x32_f16: lane 16 g + r holds 8 weights of row r.  The inputs ride on the rows of operand A in three f16
// parts (11 bits each: all 24 bits of an f32), scaled by the power of two that takes the largest magnitude of their 256
// columns to [2^14, 2^15): token t's parts are rows 4 t .. 4 t + 2, so its three sums come out in one lane (16 t + r) and the
// block's scale is one multiply-add there.  Products are exact and sums are f32; an integer is decoded once for up to 8 inputs
// (1.3 vector instructions a Q8_0 weight, 4 an IQ3_S one, where the vector unit alone took 2 and 8 and one more a token).
// Weights go from memory straight into registers, 16 rows of 8 or 16 bytes a load, a 256-column chunk ahead of the products;
// the parts of a chunk lie in a strip of LDS of the wave's own, so nothing in the loop waits for another wave.
// Measured: Q8_0, 8201 rows of 3072, 5 inputs: 25 us where the vector unit took 41; what bounds it is how its loads meet the
// memory (the same loads alone, without a product: 12 us, 2.2 TB/s).
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef u32 u32x2b __attribute__((ext_vector_type(2), aligned(2)));   // GGUF rows are only 2-byte aligned
typedef u32 u32x4b __attribute__((ext_vector_type(4), aligned(2)));

#define GG_PITCH 264   /* f16 from one A row of a strip to the next: 256 and a shift of four banks */
#define GG_STRIP(NG) (12 * (NG) * GG_PITCH)

__device__ __forceinline__ f16x2 gg_pair(u32 v) { return __builtin_bit_cast(f16x2, v); }
__device__ __forceinline__ u32 gg_bits(f16x2 v) { return __builtin_bit_cast(u32, v); }

// A lane's share of 16 rows x 256 columns: load() of row r's chunk (r = lane % 16, g = lane / 16), then products().
struct GgQ8 {
    static constexpr u32 QK = 32, BB = 34, CHUNK = 272;   // bytes of a 256-column chunk
    static constexpr bool grid = false;
    u32 q[8][2], d[8];
    __device__ __forceinline__ void load(const u8* __restrict__ p, u32 blocks, u32 g) {   // blocks: 32-blocks the chunk has (8, or fewer at the row's end)
#pragma unroll
        for (int b = 0; b < 8; b++) {
            const u8* a = p + 34 * min((u32) b, blocks - 1);
            const u32x2b v = *(const u32x2b*) (a + 2 + 8 * g);
            q[b][0] = v[0];
            q[b][1] = v[1];
            d[b] = *(const u16*) a;
        }
    }
    // four codes to f16: 0x6400 | (code ^ 0x80) is 1024 + code + 128
    static __device__ __forceinline__ void codes(u32 v, u32& lo, u32& hi) {
        const u32 t = v ^ 0x80808080u;
        const f16x2 k = {(_Float16) -1152.0f, (_Float16) -1152.0f};
        lo = gg_bits(gg_pair(__builtin_amdgcn_perm(0x64646464u, t, 0x04010400u)) + k);
        hi = gg_bits(gg_pair(__builtin_amdgcn_perm(0x64646464u, t, 0x04030402u)) + k);
    }
    // out[g] += the chunk's sums of the lane's token 4 g + lane / 16 and row lane % 16, in units of the inputs' scale
    template <int NG>
    __device__ __forceinline__ void products(const u16* __restrict__ strip, u32 blocks, u32 lane, const u32*, float (&out)[NG]) const {
        const u32 g = lane >> 4, ar = lane & 15;
        const u16* a = strip + ((ar >> 2) * 3 + min(ar & 3, 2u)) * GG_PITCH + 8 * g;
#pragma unroll
        for (int b = 0; b < 8; b++) {
            if ((u32) b < blocks) {
                u32x4 w;
                u32 t0, t1, t2, t3;
                codes(q[b][0], t0, t1);
                codes(q[b][1], t2, t3);
                w = u32x4{t0, t1, t2, t3};
                const float dd = f16_to_f32((u16) d[b]);
#pragma unroll
                for (int G = 0; G < NG; G++) {
                    const u32x4 av = *(const u32x4*) (a + 12 * G * GG_PITCH + 32 * b);
                    const f32x4 s = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, av), __builtin_bit_cast(f16x8, w), f32x4{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
                    out[G] = __builtin_fmaf((s[0] + s[1]) + s[2], dd, out[G]);
                }
            }
        }
    }
};
// IQ3_S: lane group g takes the sub-blocks 2 g and 2 g + 1 of the 256-block, 64 weights that lie together: the k order of the
// eight matrix instructions is the lane's own (instruction i: columns 64 g + 8 i ..), the same on both operands.
struct GgIq3 {
    static constexpr u32 QK = 256, BB = 110, CHUNK = 110;
    static constexpr bool grid = true;
    u32 qs[4], sg[2], qh, sc, d;
    __device__ __forceinline__ void load(const u8* __restrict__ p, u32, u32 g) {
        const u32x4b v = *(const u32x4b*) (p + 2 + 16 * g);
        const u32x2b s = *(const u32x2b*) (p + 74 + 8 * g);
#pragma unroll
        for (int i = 0; i < 4; i++) qs[i] = v[i];
        sg[0] = s[0];
        sg[1] = s[1];
        qh = *(const u16*) (p + 66 + 2 * g);
        sc = p[106 + g];
        d = *(const u16*) p;
    }
    template <int NG>
    __device__ __forceinline__ void products(const u16* __restrict__ strip, u32, u32 lane, const u32* table, float (&out)[NG]) const {
        const u32 g = lane >> 4, ar = lane & 15;
        const u16* a = strip + ((ar >> 2) * 3 + min(ar & 3, 2u)) * GG_PITCH + 64 * g;
        f32x4 s[NG];
#pragma unroll
        for (int G = 0; G < NG; G++) s[G] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int h = 0; h < 2; h++) {
            // (1024 + magnitude) * scale - 1024 * scale = magnitude * scale, exact and in one packed multiply-add
            const _Float16 sf = (_Float16) (float) (1 + 2 * ((sc >> (4 * h)) & 15u));
            const f16x2 sp = {sf, sf}, sn = {(_Float16) (-1024.0f * (float) sf), (_Float16) (-1024.0f * (float) sf)};
#pragma unroll
            for (int i = 0; i < 4; i++) {
                u32x4 w;
#pragma unroll
                for (int e = 0; e < 2; e++) {
                    const int j = 8 * h + 2 * i + e;   // grid entry of the lane's 16
                    const u32 at = (__builtin_amdgcn_ubfe(qs[j >> 2], 8 * (j & 3), 8) << 2) | (__builtin_amdgcn_ubfe(qh, j, 1) << 10);
                    const u32 m = *(const u32*) ((const u8*) table + at);
                    const u32 n = __builtin_amdgcn_ubfe(sg[j >> 3], 4 * (j & 7), 4);
                    const f16x2 lo = __builtin_elementwise_fma(gg_pair(__builtin_amdgcn_perm(0x64646464u, m, 0x04010400u)), sp, sn);
                    const f16x2 hi = __builtin_elementwise_fma(gg_pair(__builtin_amdgcn_perm(0x64646464u, m, 0x04030402u)), sp, sn);
                    // a set sign bit flips its value's sign: bits 0, 1 to bits 15, 31 of the pair, bits 2, 3 of the other
                    w[2 * e] = gg_bits(lo) ^ ((n * 0x40008000u) & 0x80008000u);
                    w[2 * e + 1] = gg_bits(hi) ^ (((n >> 2) * 0x40008000u) & 0x80008000u);
                }
#pragma unroll
                for (int G = 0; G < NG; G++) {
                    const u32x4 av = *(const u32x4*) (a + 12 * G * GG_PITCH + 32 * h + 8 * i);
                    s[G] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, av), __builtin_bit_cast(f16x8, w), s[G], 0, 0, 0);
                }
            }
        }
        const float dd = f16_to_f32((u16) d);
#pragma unroll
        for (int G = 0; G < NG; G++) out[G] = __builtin_fmaf((s[G][0] + s[G][1]) + s[G][2], dd, out[G]);
    }
};

// The parts of 256 columns of the inputs into the wave's strip; v[r]: the lane's four columns of input r.  s_iv[r] undoes the scale.
template <int NMAX>
__device__ __forceinline__ void gg_split(const f32x4 (&v)[NMAX], u32 n, u16* strip, float* s_iv, u32 lane) {
#pragma unroll
    for (int r = 0; r < NMAX; r++) {
        if ((u32) r < n) {
            const float mx = wave_max_f32(fmaxf(fmaxf(__builtin_fabsf(v[r][0]), __builtin_fabsf(v[r][1])), fmaxf(__builtin_fabsf(v[r][2]), __builtin_fabsf(v[r][3]))));
            float scale, iv;
            pow2_scale_of(f32_bits(mx), scale, iv);
            if (lane == 0) s_iv[r] = iv;
            u32 part[3][2];
#pragma unroll
            for (int i = 0; i < 2; i++) {
                const float a = v[r][2 * i] * scale, b = v[r][2 * i + 1] * scale;
                const _Float16 ah = (_Float16) a, bh = (_Float16) b;
                const float a1 = a - (float) ah, b1 = b - (float) bh;
                const _Float16 am = (_Float16) a1, bm = (_Float16) b1;
                part[0][i] = gg_bits(f16x2{ah, bh});
                part[1][i] = gg_bits(f16x2{am, bm});
                part[2][i] = gg_bits(f16x2{(_Float16) (a1 - (float) am), (_Float16) (b1 - (float) bm)});
            }
#pragma unroll
            for (int p = 0; p < 3; p++) *(uint2*) (strip + (3 * r + p) * GG_PITCH + 4 * lane) = uint2{part[p][0], part[p][1]};
        }
    }
}

// A wave's products: its chunks c0, c0 + step, .. of the row (256 columns each) of RT tiles of 16 rows; wrow[t]: the lane's row of
// tile t; row(r): input r's first column.  tot[t][G]: row lane % 16 of the tile, token 4 G + lane / 16.
template <class F, int NG, int RT, class Row>
__device__ __forceinline__ void gg_wave(const u8* const (&wrow)[RT], u32 cols, u32 c0, u32 step, Row row, u32 n, u16* strip, float* s_iv, const u32* table, u32 lane,
                                        float (&tot)[RT][NG]) {
    constexpr int NMAX = 4 * NG;
    const u32 nc = (cols + 255) / 256, g = lane >> 4;
    auto blocks = [&](u32 c) { return min(8u, cols / 32 - 8 * c); };
#pragma unroll
    for (int t = 0; t < RT; t++)
#pragma unroll
        for (int G = 0; G < NG; G++) tot[t][G] = 0.0f;
    if (c0 >= nc) return;
    F cur[RT], nxt[RT];
    f32x4 v[NMAX];
    auto inputs = [&](u32 c) {
#pragma unroll
        for (int r = 0; r < NMAX; r++) {
            v[r] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            if ((u32) r < n && 256 * c + 4 * lane < cols) v[r] = *(const f32x4*) (row((u32) r) + 256 * c + 4 * lane);
        }
    };
    inputs(c0);
#pragma unroll
    for (int t = 0; t < RT; t++) cur[t].load(wrow[t] + (u64) c0 * F::CHUNK, blocks(c0), g);
    for (u32 c = c0; c < nc; c += step) {
        const u32 cn = min(c + step, nc - 1);
        gg_split<NMAX>(v, n, strip, s_iv, lane);
        inputs(cn);
#pragma unroll
        for (int t = 0; t < RT; t++) nxt[t].load(wrow[t] + (u64) cn * F::CHUNK, blocks(cn), g);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
        for (int t = 0; t < RT; t++) {
            float out[NG];
#pragma unroll
            for (int G = 0; G < NG; G++) out[G] = 0.0f;
            cur[t].template products<NG>(strip, blocks(c), lane, table, out);
#pragma unroll
            for (int G = 0; G < NG; G++) tot[t][G] = __builtin_fmaf(out[G], s_iv[4 * G + g], tot[t][G]);
        }
        __builtin_amdgcn_wave_barrier();   // the strip is read before the next chunk's parts go there (LDS is in order within a wave)
#pragma unroll
        for (int t = 0; t < RT; t++) cur[t] = nxt[t];
    }
}

// Where a wave leaves its 2 NG 64 sums for the workgroup: in its strip, which it is done with.
template <int NG>
__device__ __forceinline__ float* gg_red(u16 (*strip)[GG_STRIP(NG)], u32 wave) { return (float*) strip[wave]; }

__device__ __forceinline__ void gg_table(u32* table) {
    for (u32 i = threadIdx.x; i < 512; i += blockDim.x) table[i] = IQ3S_GRID[i];
}

// y_j = W x_j, j < m: x rows xs floats apart, y rows ys apart (matvec_cols_*, kernels/matvec.cu:677).  A workgroup takes 32 rows
// for every 4 / ks waves of its 4, ks waves share a row's chunks (1, 2 or 4 by the number of chunks alone: the sums' order, so
// the bits, do not depend on m).  grid = ceil(rows / (128 / ks)), block 256.
template <class F, int NG>
__device__ __forceinline__ void gg_cols(const u8* __restrict__ w, const float* __restrict__ x, u32 xs, float* __restrict__ y, u32 ys, u32 rows, u32 cols, u32 m, u32 ks) {
    __shared__ __attribute__((aligned(16))) u16 strip[4][GG_STRIP(NG)];
    __shared__ float s_iv[4][4 * NG];
    __shared__ u32 table[F::grid ? 512 : 1];
    const u32 wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const u32 kw = wave & (ks - 1), first = (blockIdx.x * (4 / ks) + wave / ks) * 32;
    const u32 rb = cols / F::QK * F::BB;
    const u8* wrow[2];
#pragma unroll
    for (int t = 0; t < 2; t++) wrow[t] = w + (u64) min(first + 16 * t + (lane & 15), rows - 1) * rb;
    if constexpr (F::grid) {
        gg_table(table);
        __syncthreads();
    }
    float tot[2][NG];
    gg_wave<F, NG, 2>(wrow, cols, kw, ks, [&](u32 r) { return x + (u64) r * xs; }, m, strip[wave], s_iv[wave], table, lane, tot);
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
        for (int G = 0; G < NG; G++) gg_red<NG>(strip, wave)[(t * NG + G) * 64 + lane] = tot[t][G];
    __syncthreads();
    for (u32 i = threadIdx.x; i < 4 / ks * 2 * NG * 64; i += 256) {
        const u32 q = i / (2 * NG * 64), p = i % (2 * NG * 64), t = p / (NG * 64), G = p / 64 % NG, l = p & 63;
        float s = gg_red<NG>(strip, q * ks)[p];
        for (u32 k = 1; k < ks; k++) s += gg_red<NG>(strip, q * ks + k)[p];
        const u32 r = (blockIdx.x * (4 / ks) + q) * 32 + 16 * t + (l & 15), j = 4 * G + (l >> 4);
        if (r < rows && j < m) y[(u64) j * ys + r] = s;
    }
}
extern "C" __global__ void __launch_bounds__(256, 3) matvec_cols_q8_0(const u8* w, const float* x, u32 xs, float* y, u32 ys, u32 rows, u32 cols, u32 m, u32 ks) {
    gg_cols<GgQ8, 1>(w, x, xs, y, ys, rows, cols, m, ks);
}
extern "C" __global__ void __launch_bounds__(256, 3) matvec_cols_w_q8_0(const u8* w, const float* x, u32 xs, float* y, u32 ys, u32 rows, u32 cols, u32 m, u32 ks) {
    gg_cols<GgQ8, 2>(w, x, xs, y, ys, rows, cols, m, ks);
}
extern "C" __global__ void __launch_bounds__(256, 3) matvec_cols_iq3_s(const u8* w, const float* x, u32 xs, float* y, u32 ys, u32 rows, u32 cols, u32 m, u32 ks) {
    gg_cols<GgIq3, 1>(w, x, xs, y, ys, rows, cols, m, ks);
}
extern "C" __global__ void __launch_bounds__(256, 3) matvec_cols_w_iq3_s(const u8* w, const float* x, u32 xs, float* y, u32 ys, u32 rows, u32 cols, u32 m, u32 ks) {
    gg_cols<GgIq3, 2>(w, x, xs, y, ys, rows, cols, m, ks);
}
