// Matrix-vector products over GGUF row-major quantized matrices (Q8_0, IQ3_S) for 1..4 inputs at a time.
//
// Shape of every fast kernel here: a workgroup of 256 threads (4 waves of 64) owns `rpb` consecutive rows.  The rows'
// bytes are one contiguous span of the matrix, so the workgroup streams them from HBM with 16-byte loads, lane after
// lane, into LDS; nothing about the 34-byte (Q8_0) or 110-byte (IQ3_S) block boundaries matters to the HBM side.  Each
// lane then decodes one unit of 32 weights from LDS against inputs it holds in registers, and a segment of lanes is
// summed with wave shuffles.  Follows the semantics of the reference's matvec_cols_* / matvec_grouped_* kernels
// (kernels/matvec.cu:677-756, 1576-1677): y_j = W x_j with the weights decoded once for all inputs.

struct Q80 {
    static constexpr u32 QK = 32, BB = 34;
};
struct IQ3S {
    static constexpr u32 QK = 256, BB = 110;
};

// ------------------------------------------------------------------------------------------------ reference kernels
// One wave a row, a lane every 64th weight, each weight decoded on its own from global memory: correct for any column
// count that is a whole number of blocks; the kernel GpuBackend::matvec uses (crates/shadowzero-cuda/src/backend.rs:57-101, matvec.cu:7-32).
__device__ __forceinline__ float q8_0_at(const u8* row, u32 i) {
    const u8* b = row + (u64) (i / 32) * 34;
    const float d = f16_to_f32((u16) (b[0] | (b[1] << 8)));
    return d * (float) (i8) b[2 + (i % 32)];
}

__device__ __forceinline__ float iq3_s_at(const u8* row, u32 i) {
    const u8* b = row + (u64) (i / 256) * 110;
    const u32 e = i % 256, j = e / 4, g = e / 32;
    const float d = f16_to_f32((u16) (b[0] | (b[1] << 8)));
    const u32 idx = b[2 + j] | (((b[66 + j / 8] >> (j % 8)) & 1u) << 8);
    const u32 s = (b[106 + g / 2] >> (4 * (g % 2))) & 0x0f;
    const float db = d * (float) (1 + 2 * s);
    const float grid = (float) ((IQ3S_GRID[idx] >> (8 * (e % 4))) & 0xff);
    const float sg = ((b[74 + e / 8] >> (e % 8)) & 1) ? -1.0f : 1.0f;
    return db * grid * sg;
}

extern "C" __global__ void __launch_bounds__(256) matvec_q8_0(const u8* w, const float* x, float* y, u32 rows, u32 cols) {
    const u32 r = blockIdx.x * 4 + threadIdx.x / 64, lane = threadIdx.x % 64;
    if (r >= rows) return;
    const u8* row = w + (u64) r * (cols / 32 * 34);
    float acc = 0.0f;
    for (u32 i = lane; i < cols; i += 64) acc = __builtin_fmaf(q8_0_at(row, i), x[i], acc);
    acc = seg_sum<64>(acc, lane);
    if (lane == 0) y[r] = acc;
}

extern "C" __global__ void __launch_bounds__(256) matvec_iq3_s(const u8* w, const float* x, float* y, u32 rows, u32 cols) {
    const u32 r = blockIdx.x * 4 + threadIdx.x / 64, lane = threadIdx.x % 64;
    if (r >= rows) return;
    const u8* row = w + (u64) r * (cols / 256 * 110);
    float acc = 0.0f;
    for (u32 i = lane; i < cols; i += 64) acc = __builtin_fmaf(iq3_s_at(row, i), x[i], acc);
    acc = seg_sum<64>(acc, lane);
    if (lane == 0) y[r] = acc;
}

// Whole blocks to f32, a thread a weight, in the CPU reference's operation order (quant.rs:148-179): bit-exact test hooks.
extern "C" __global__ void __launch_bounds__(256) dequant_q8_0(const u8* w, float* out, u64 n) {
    const u64 i = (u64) blockIdx.x * 256 + threadIdx.x;
    if (i < n) out[i] = q8_0_at(w + (i / 32) * 34, (u32) (i % 32));
}

extern "C" __global__ void __launch_bounds__(256) dequant_iq3_s(const u8* w, float* out, u64 n) {
    const u64 i = (u64) blockIdx.x * 256 + threadIdx.x;
    if (i < n) out[i] = iq3_s_at(w + (i / 256) * 110, (u32) (i % 256));
}

// ------------------------------------------------------------------------------------------------------ LDS staging
extern __shared__ u32 sz_dyn_lds[];

// Copies bytes [g0, g0 + span) of global memory to LDS so that byte g0 lands at LDS byte (g0 & 15): whole 16-byte
// chunks, one per thread per step, except a first or last chunk that would reach outside the span, which is read
// byte by byte so that the kernel never touches memory outside the matrix.
__device__ __forceinline__ u32 stage_span(const u8* g0, u32 span, u32 tid) {
    const u32 head = (u32) ((u64) g0 & 15);
    const u8* a0 = g0 - head;
    const u32 total = head + span;
    const u32 nchunks = (total + 15) / 16;
    if (head == 0 && total % 16 == 0) {
        // the usual case, whole chunks only: four a thread a round, their loads all in flight before the first store (a
        // load-store loop takes a memory round trip a chunk); a thread past the end reads the last chunk again and drops it
        for (u32 c0 = 0; c0 < nchunks; c0 += 1024) {
            u32x4 v[4];
#pragma unroll
            for (int i = 0; i < 4; i++) v[i] = *(const u32x4*) (a0 + (u64) min(c0 + tid + 256 * i, nchunks - 1) * 16);
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const u32 c = c0 + tid + 256 * i;
                if (c < nchunks) ((u32x4*) sz_dyn_lds)[c] = v[i];
            }
        }
        return head;
    }
    for (u32 c = tid; c < nchunks; c += 256) {
        u32x4 v;
        if ((c == 0 && head != 0) || (c * 16 + 16 > total)) {
            u32 w[4] = {0, 0, 0, 0};
            for (u32 b = 0; b < 16; b++) {
                const u32 idx = c * 16 + b;
                if (idx >= head && idx < total) w[b / 4] |= (u32) a0[idx] << (8 * (b % 4));
            }
            v = u32x4{w[0], w[1], w[2], w[3]};
        } else {
            v = *(const u32x4*) (a0 + c * 16);
        }
        ((u32x4*) sz_dyn_lds)[c] = v;
    }
    return head;
}

__device__ __forceinline__ u32 lds_u8(u32 o) { return ((const u8*) sz_dyn_lds)[o]; }
__device__ __forceinline__ u32 lds_u16(u32 o) { return ((const u16*) sz_dyn_lds)[o >> 1]; }   // o even
__device__ __forceinline__ u32 lds_u32(u32 o) { return sz_dyn_lds[o >> 2]; }                  // o multiple of 4

// ------------------------------------------------------------------------------------------------------- unit dots
// out[j] = sum over the unit's 32 weights of w_i * x[i][j], the block scale included.  `o` is the LDS byte offset of the
// unit's row; `u` the unit's index in the row.
template <int M>
__device__ __forceinline__ void unit_dot_q8_0(u32 o, u32 u, const float (&x)[32][M], float (&out)[M]) {
    const u32 b = o + 34 * u;
    const float d = f16_to_f32((u16) lds_u16(b));
    const u32 q0 = b + 2;                       // the 32 codes; q0 is 0 or 2 modulo 4
    const u32 sh = (q0 & 3) * 8;
    const u32 a = q0 & ~3u;
    u32 dw[9];
#pragma unroll
    for (int i = 0; i < 9; i++) dw[i] = lds_u32(a + 4 * i);
    float acc[M];
#pragma unroll
    for (int j = 0; j < M; j++) acc[j] = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const u32 q = __builtin_amdgcn_alignbit(dw[i + 1], dw[i], sh);
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const float w = (float) (i8) (q >> (8 * k));
#pragma unroll
            for (int j = 0; j < M; j++) acc[j] = __builtin_fmaf(w, x[4 * i + k][j], acc[j]);
        }
    }
#pragma unroll
    for (int j = 0; j < M; j++) out[j] = d * acc[j];
}

__shared__ u32 sz_iq3s_grid[512];

// The signs of four weights (bits 0..3 of n) applied to their packed magnitudes (four bytes, each at most 15): a set bit
// negates its byte.  n * 0x00204081 puts bit i of n at bit 8 i (and others in between), the mask leaves 0 or 1 a byte, times 255 is
// 0x00 or 0xff a byte, and (m ^ ff) + 1 = -m byte by byte (no carries: the magnitudes are below 128, and -m + ... stays in its byte).
__device__ __forceinline__ u32 iq3s_signed4(u32 mags, u32 n) {
    const u32 one = (n * 0x00204081u) & 0x01010101u;
    return (mags ^ (one * 255u)) + one;
}

template <int M>
__device__ __forceinline__ void unit_dot_iq3_s(u32 o, u32 u, const float (&x)[32][M], float (&out)[M]) {
    const u32 b = o + 110 * (u >> 3), g = u & 7;
    const float d = f16_to_f32((u16) lds_u16(b));
    const u32 qo = b + 2 + 8 * g;
    const u32 qs0 = lds_u16(qo) | (lds_u16(qo + 2) << 16), qs1 = lds_u16(qo + 4) | (lds_u16(qo + 6) << 16);
    const u32 qh = lds_u8(b + 66 + g);
    const u32 so = b + 74 + 4 * g;
    const u32 signs = lds_u16(so) | (lds_u16(so + 2) << 16);
    const u32 sc = (lds_u8(b + 106 + (g >> 1)) >> (4 * (g & 1))) & 0x0f;
    const float db = d * (float) (1 + 2 * sc);
    float acc[M];
#pragma unroll
    for (int j = 0; j < M; j++) acc[j] = 0.0f;
#pragma unroll
    for (int jj = 0; jj < 8; jj++) {
        // the table's byte offset: 4 * (index byte | high bit << 8), from two bit-field extracts, a shift and a shift-or
        const u32 at = (__builtin_amdgcn_ubfe(jj < 4 ? qs0 : qs1, 8 * (jj & 3), 8) << 2) | (__builtin_amdgcn_ubfe(qh, jj, 1) << 10);
        const u32 grid = *(const u32*) ((const u8*) sz_iq3s_grid + at);
        const u32 sg = iq3s_signed4(grid, __builtin_amdgcn_ubfe(signs, 4 * jj, 4));
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int i = 4 * jj + k;
            const float w = (float) (i8) (sg >> (8 * k));        // one sign-extending byte conversion
#pragma unroll
            for (int j = 0; j < M; j++) acc[j] = __builtin_fmaf(w, x[i][j], acc[j]);
        }
    }
#pragma unroll
    for (int j = 0; j < M; j++) out[j] = db * acc[j];
}

template <class F, int M>
__device__ __forceinline__ void unit_dot(u32 o, u32 u, const float (&x)[32][M], float (&out)[M]) {
    if constexpr (F::BB == 34) unit_dot_q8_0<M>(o, u, x, out);
    else unit_dot_iq3_s<M>(o, u, x, out);
}

// An input row shared by a workgroup through LDS: the 32 inputs of unit u start at float 36 u
// (a lane reads them with eight 16-byte LDS loads; the 4 floats of padding spread the units over the banks).  Reading a
// unit's 128 bytes from global memory lane by lane instead costs the texture path a cache line a lane per load.
constexpr u32 XU_PITCH = 36;

__device__ __forceinline__ void unit_from_lds(const float* xs, u32 u, float (&x)[32][1]) {
    const f32x4* p = (const f32x4*) (xs + u * XU_PITCH);
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const f32x4 v = p[i];
        x[4 * i][0] = v.x;
        x[4 * i + 1][0] = v.y;
        x[4 * i + 2][0] = v.z;
        x[4 * i + 3][0] = v.w;
    }
}

// ---------------------------------------------------------------------------------------------------- the row kernel
// rows_body for rows of more than 64 units (rpb <= 16: at most 4 rows a wave).  The inputs come in column chunks of 64
// units: the workgroup brings chunk c of every input into LDS (s_in, as for short rows), every lane takes its unit of
// it into registers and adds the unit's product to the running sums of the wave's rows, chunk after chunk in column order.
template <class F, int M, class After>
__device__ __forceinline__ void rows_wide(const u8* __restrict__ w, u32 rows, u32 cols, u32 rpb, const float* (&xp)[M], float* (&yp)[M],
                                          float* res, After after_chunk, float (*s_in)[64 * XU_PITCH]) {
    const u32 tid = threadIdx.x, wave = tid / 64, lane = tid % 64;
    const u32 rb = cols / F::QK * F::BB, U = cols / 32, NC = (U + 63) / 64;
    const u32 nchunks = (rows + rpb - 1) / rpb;
    for (u32 chunk = blockIdx.x; chunk < nchunks; chunk += gridDim.x) {
        const u32 r0 = chunk * rpb;
        const u32 nrows = min(rpb, rows - r0);
        const u32 head = stage_span(w + (u64) r0 * rb, nrows * rb, tid);
        float tot[4][M];
#pragma unroll
        for (int r = 0; r < 4; r++)
#pragma unroll
            for (int j = 0; j < M; j++) tot[r][j] = 0.0f;
        for (u32 c = 0; c < NC; c++) {
            f32x4 piece[M][2];
#pragma unroll
            for (int j = 0; j < M; j++)
#pragma unroll
                for (int h = 0; h < 2; h++) piece[j][h] = ((const f32x4*) xp[j])[min(c * 512 + tid + 256 * h, cols / 4 - 1)];
            if (c) __syncthreads();               // every lane has taken its unit of the chunk before
#pragma unroll
            for (int j = 0; j < M; j++)
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    const u32 i = tid + 256 * h;
                    *(f32x4*) (s_in[j] + (i / 8) * XU_PITCH + (i % 8) * 4) = piece[j][h];
                }
            __syncthreads();                      // the chunk (and, the first time, the staged rows)
            const u32 un = c * 64 + lane;
            if (un < U) {
                float x[32][M];
#pragma unroll
                for (int j = 0; j < M; j++) {
                    const f32x4* p = (const f32x4*) (s_in[j] + lane * XU_PITCH);
#pragma unroll
                    for (int i = 0; i < 8; i++) {
                        const f32x4 v = p[i];
                        x[4 * i][j] = v.x;
                        x[4 * i + 1][j] = v.y;
                        x[4 * i + 2][j] = v.z;
                        x[4 * i + 3][j] = v.w;
                    }
                }
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const u32 lr = wave + 4 * r;
                    if (lr < nrows) {
                        float part[M];
                        unit_dot<F, M>(head + lr * rb, un, x, part);
#pragma unroll
                        for (int j = 0; j < M; j++) tot[r][j] += part[j];
                    }
                }
            }
        }
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const u32 lr = wave + 4 * r;
#pragma unroll
            for (int j = 0; j < M; j++) tot[r][j] = seg_sum<64>(tot[r][j], lane);
            if (lane == 0 && lr < nrows) {
#pragma unroll
                for (int j = 0; j < M; j++) {
                    if (yp[j]) yp[j][r0 + lr] = tot[r][j];
                    if (res) res[lr * 4 + j] = tot[r][j];
                }
            }
        }
        __syncthreads();          // every wave is done with the staged bytes and the inputs (and res is complete)
        if (res) {
            after_chunk(r0, nrows);
            __syncthreads();
        }
    }
}

// Row chunks blockIdx.x, blockIdx.x + gridDim.x, .. (rpb rows each) of `w` against M inputs: the inputs are read into
// registers once per workgroup, then every chunk is staged and decoded.  Results go through yp to global memory and, when
// `res` is given, to res[local row * 4 + j] in LDS, after which after_chunk(first row, rows) runs on every thread between
// two barriers.  cols is a multiple of 32 (and of the format's block).
template <class F, int M, class After>
__device__ __forceinline__ void rows_body(const u8* __restrict__ w, u32 rows, u32 cols, u32 rpb, const float* (&xp)[M],
                                          float* (&yp)[M], float* res, After after_chunk) {
    const u32 tid = threadIdx.x, wave = tid / 64, lane = tid % 64;
    const u32 rb = cols / F::QK * F::BB;
    if constexpr (F::BB == 110) {
        for (u32 i = tid; i < 512; i += 256) sz_iq3s_grid[i] = IQ3S_GRID[i];
    }
    const u32 U = cols / 32;
    u32 UL = 64;                          // lanes a row takes in a wave: the units of a row of fewer than 64, rounded up to a power of two
    if (U < 64) {
        UL = 1;
        while (UL < U) UL *= 2;
    }
    const u32 RG = 64 / UL;               // rows side by side in a wave
    const u32 NC = (U + UL - 1) / UL;     // column chunks of UL units; lanes past the row's last unit add nothing
    const u32 sub = lane / UL, ul = lane % UL;
    float x[32][M];
    // the workgroup reads the inputs with whole-line loads and hands them out through LDS
    __shared__ __attribute__((aligned(16))) float s_in[M][64 * XU_PITCH];
    if (NC != 1) {
        rows_wide<F, M>(w, rows, cols, rpb, xp, yp, res, after_chunk, s_in);
        return;
    }
    f32x4 piece[M][2];
#pragma unroll
    for (int j = 0; j < M; j++)
#pragma unroll
        for (int h = 0; h < 2; h++) piece[j][h] = ((const f32x4*) xp[j])[min(tid + 256 * h, cols / 4 - 1)];
    bool first = true;
    const u32 nchunks = (rows + rpb - 1) / rpb;
    for (u32 chunk = blockIdx.x; chunk < nchunks; chunk += gridDim.x) {
        const u32 r0 = chunk * rpb;
        const u32 nrows = min(rpb, rows - r0);
        const u32 head = stage_span(w + (u64) r0 * rb, nrows * rb, tid);
        if (first) {
#pragma unroll
            for (int j = 0; j < M; j++)
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    const u32 i = tid + 256 * h;
                    if (i < cols / 4) *(f32x4*) (s_in[j] + (i / 8) * XU_PITCH + (i % 8) * 4) = piece[j][h];
                }
        }
        __syncthreads();
        if (first) {
            first = false;
#pragma unroll
            for (int j = 0; j < M; j++) {
                const f32x4* p = (const f32x4*) (s_in[j] + ul * XU_PITCH);
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    const f32x4 v = p[i];
                    x[4 * i][j] = v.x;
                    x[4 * i + 1][j] = v.y;
                    x[4 * i + 2][j] = v.z;
                    x[4 * i + 3][j] = v.w;
                }
            }
        }
        for (u32 lr = wave * RG + sub; lr < rpb; lr += 4 * RG) {   // lr < rpb for every lane of a wave alike, or for none
            float tot[M];
#pragma unroll
            for (int j = 0; j < M; j++) tot[j] = 0.0f;
            if (lr < nrows && ul < U) unit_dot<F, M>(head + lr * rb, ul, x, tot);
#pragma unroll
            for (int j = 0; j < M; j++) tot[j] = seg_sum_rt(tot[j], UL, lane);
            if (ul == 0 && lr < nrows) {
#pragma unroll
                for (int j = 0; j < M; j++) {
                    if (yp[j]) yp[j][r0 + lr] = tot[j];
                    if (res) res[lr * 4 + j] = tot[j];
                }
            }
        }
        __syncthreads();          // every wave is done with the staged bytes (and res is complete)
        if (res) {
            after_chunk(r0, nrows);
            __syncthreads();
        }
    }
}

struct NoAfter {
    __device__ __forceinline__ void operator()(u32, u32) const {}
};

// y = W x for the one input of GpuBackend::matvec: with a single input there is no decoded weight to share, so the vector unit alone
// (no parts of the input to make first) answers a small product sooner than the matrix cores: 4.1 us from begin to end for 1024
// rows of 2048 Q8_0 columns where matvec_cols_q8_0 takes 4.5, 8.4 and 9.5 for 2048 x 8192 (IQ3_S 4.3 and 5.3, 8.0 and 10.3; for
// 8201 rows of 3072 it is 11.4 and 9.5).  matvec_cols has one form for every number of inputs all the same: an input's bits
// must not depend on what it is batched with, and these sums are in another order.  grid = ceil(rows / rpb), block 256, dynamic
// LDS rpb * row bytes + 32.
template <class F>
__device__ __forceinline__ void one_kernel(const u8* w, const float* x, float* y, u32 rows, u32 cols, u32 rpb) {
    const float* xp[1] = {x};
    float* yp[1] = {y};
    rows_body<F, 1>(w, rows, cols, rpb, xp, yp, nullptr, NoAfter());
}
extern "C" __global__ void __launch_bounds__(256) matvec_one_q8_0(const u8* w, const float* x, float* y, u32 rows, u32 cols, u32 rpb) {
    one_kernel<Q80>(w, x, y, rows, cols, rpb);
}
extern "C" __global__ void __launch_bounds__(256) matvec_one_iq3_s(const u8* w, const float* x, float* y, u32 rows, u32 cols, u32 rpb) {
    one_kernel<IQ3S>(w, x, y, rows, cols, rpb);
}

template <class F, class After>
__device__ __forceinline__ void rows_dispatch(const u8* w, u32 rows, u32 cols, u32 rpb, u32 n, const float* (&xp)[4],
                                              float* (&yp)[4], float* res, After after) {
    if (n == 1) {
        const float* x1[1] = {xp[0]};
        float* y1[1] = {yp[0]};
        rows_body<F, 1>(w, rows, cols, rpb, x1, y1, res, after);
    } else if (n == 2) {
        const float* x2[2] = {xp[0], xp[1]};
        float* y2[2] = {yp[0], yp[1]};
        rows_body<F, 2>(w, rows, cols, rpb, x2, y2, res, after);
    } else if (n >= 3) {
        rows_body<F, 4>(w, rows, cols, rpb, xp, yp, res, after);
    }
}

// Group g = blockIdx.y: matrix wtab[g] (device address), record gtab[17 g] = {n <= 4 (0: unused slot), xi[8], yi[8]};
// y[yi[j]] = W x[xi[j]] (matvec.cu:1576-1677).  grid = (ceil(rows / rpb), groups).
template <class F>
__device__ __forceinline__ void grouped_kernel(const u64* wtab, const u32* gtab, const float* x, u32 xs, float* y, u32 ys, u32 rows,
                                               u32 cols, u32 rpb) {
    const u32* rec = gtab + 17 * (u64) blockIdx.y;
    const u32 n = min(rec[0], 4u);
    if (n == 0) return;
    const u8* w = (const u8*) wtab[blockIdx.y];
    const float* xp[4];
    float* yp[4];
    for (u32 j = 0; j < 4; j++) {
        const u32 jj = j < n ? j : 0;
        xp[j] = x + (u64) rec[1 + jj] * xs;
        yp[j] = j < n ? y + (u64) rec[9 + jj] * ys : nullptr;
    }
    rows_dispatch<F>(w, rows, cols, rpb, n, xp, yp, nullptr, NoAfter());
}

extern "C" __global__ void __launch_bounds__(256) matvec_grouped_q8_0(const u64* wtab, const u32* gtab, const float* x, u32 xs, float* y,
                                                                      u32 ys, u32 rows, u32 cols, u32 rpb) {
    grouped_kernel<Q80>(wtab, gtab, x, xs, y, ys, rows, cols, rpb);
}

extern "C" __global__ void __launch_bounds__(256) matvec_grouped_iq3_s(const u64* wtab, const u32* gtab, const float* x, u32 xs, float* y,
                                                                       u32 ys, u32 rows, u32 cols, u32 rpb) {
    grouped_kernel<IQ3S>(wtab, gtab, x, xs, y, ys, rows, cols, rpb);
}

// Rows [rpb blockIdx.x, +rpb) of w against the workgroup's inputs in LDS, for a launch with one chunk a workgroup and a
// row's units inside a wave (U = cols / 32 divides 64): the sums are those of rows_body with one input, bit for bit.
// Every thread has passed a barrier since xs (and the IQ3_S table) was written.
template <class F>
__device__ __forceinline__ void rows_one_chunk(const u8* w, u32 rows, u32 cols, u32 rpb, u32 head, const float* xs, float* y) {
    const u32 lane = threadIdx.x % 64, wv = threadIdx.x / 64;
    const u32 U = cols / 32, rb = cols / F::QK * F::BB;
    const u32 r0 = blockIdx.x * rpb;
    const u32 nrows = min(rpb, rows - r0);
    const u32 lg = 31u - (u32) __builtin_clz(U), RG = 64u >> lg, sub = lane >> lg, ul = lane & (U - 1);   // U divides 64: a power of two
    float x[32][1];
    unit_from_lds(xs, ul, x);
    for (u32 lr = wv * RG + sub; lr < rpb; lr += 4 * RG) {
        float tot[1] = {0.0f};
        if (lr < nrows) unit_dot<F, 1>(head + lr * rb, ul, x, tot);
        tot[0] = seg_sum_rt(tot[0], U, lane);
        if (ul == 0 && lr < nrows) y[r0 + lr] = tot[0];
    }
}

// -------------------------------------------------------------------------------------- the verify layer, GGUF experts
// A resident Q8_0 / IQ3_S layer for a verify batch (m <= 8 rows) without a plan, in the shape of the EXL3 one: the work
// items are the (token, expert) pairs themselves, one input each: pair p = j k + t of token j and rank t for p < m k, then
// the shared expert's pair m k + j of every token j.  Expert e's three matrices sit at ebase + e estride + {0, part, 2 part}
// (gate, up, down), the shared expert's at shbase + the same offsets (shbase = 0: none).
// pbuf holds u32 tidx[m k] | f32 w[m k] | u32 cnt[m]; eg holds the gate rows [S][ff] then the up rows [S][ff], S = m (k + 1).
// Every product is the single-input case of rows_body, so the numbers are those of the planned path bit for bit.

// Launch 1: routing (every workgroup of a routed pair redoes its token's selection on one of its waves; the workgroups
// with blockIdx.x == 0 of the gate half also publish tidx), then rows [rpb blockIdx.x, +rpb) of gate (sel 0) or up (sel 1).
// grid = (ceil(ff / rpb), 2 S), block 256, dynamic LDS = rpb * row bytes + 32.
template <class F>
__device__ __forceinline__ void verify_gate_up_gguf(const float* logits, u64 ebase, u64 estride, u64 shbase, u32 part, const float* u, u8* pbuf,
                                                    float* eg, u32 ne, u32 k, u32 m, u32 hidden, u32 ff, u32 rpb) {
    __shared__ u32 s_top[16];
    __shared__ double s_ex[512];   // only the exact fallback of the routing touches it
    __shared__ __attribute__((aligned(16))) float s_x[64 * XU_PITCH];
    const u32 G = m * k, S = G + m;
    const u32 wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const u32 sel = blockIdx.y / S, pair = blockIdx.y % S;
    const u32 j = pair < G ? pair / k : pair - G;
    const float* xp[1] = {u + (u64) j * hidden};
    float* yp[1] = {eg + (u64) (sel * S + pair) * ff};
    // one chunk a workgroup and a row's units inside a wave: the token's inputs go through LDS, with loads that are asked
    // for before the routing and cost it little (whole lines a wave, unlike a lane's own 128 bytes)
    const u32 U = hidden / 32;
    const bool one = U <= 64 && 64 % U == 0 && gridDim.x * rpb >= ff;
    if (one) {
        for (u32 i = threadIdx.x; i < hidden / 4; i += 256) *(f32x4*) (s_x + (i / 8) * XU_PITCH + (i % 8) * 4) = ((const f32x4*) xp[0])[i];
        if constexpr (F::BB == 110) {
            for (u32 i = threadIdx.x; i < 512; i += 256) sz_iq3s_grid[i] = IQ3S_GRID[i];
        }
    }
    const u8* w;
    if (pair < G) {
        const u32 t = pair % k;
        if (wave == ((blockIdx.x + blockIdx.y) & 3u)) {
            __builtin_amdgcn_s_setprio(3);   // every other wave of the workgroup waits for this one
            route_id_of_rank(logits + (u64) j * ne, ne, k, t, lane, s_ex, s_top);   // only s_top[t] is read
            __builtin_amdgcn_s_setprio(0);
            if (sel == 0 && blockIdx.x == 0 && lane == 0) ((u32*) pbuf)[pair] = s_top[t];
        }
        __syncthreads();
        const u32 e = s_top[t];
        if (e == 0xffffffffu) return;
        w = (const u8*) (ebase + e * estride + (u64) sel * part);
    } else {
        if (!shbase) return;
        w = (const u8*) (shbase + (u64) sel * part);
    }
    if (one) {
        const u32 rb = hidden / F::QK * F::BB, r0 = blockIdx.x * rpb;
        const u32 head = stage_span(w + (u64) r0 * rb, min(rpb, ff - r0) * rb, threadIdx.x);
        __syncthreads();       // the rows, and for the shared expert's pairs also s_x and the table
        rows_one_chunk<F>(w, ff, hidden, rpb, head, s_x, yp[0]);
        return;
    }
    rows_body<F, 1>(w, ff, hidden, rpb, xp, yp, nullptr, NoAfter());
}

// Launch 2: act = silu(gate) * up of the pair (every workgroup makes its own copy in LDS: ff values), then rows
// [rpb blockIdx.x, +rpb) of down into eo[pair][hidden].  One wave a token also computes the routing weights and the count
// for the combine.  grid = (ceil(hidden / rpb), S), block 256, dynamic LDS = rpb * row bytes + 32; ff <= 4096.
template <class F>
__device__ __forceinline__ void verify_down_gguf(const float* logits, u64 ebase, u64 estride, u64 shbase, u32 part, u8* pbuf, const float* eg,
                                                 float* eo, u32 ne, u32 k, u32 m, u32 hidden, u32 ff, u32 rpb) {
    __shared__ __attribute__((aligned(16))) float act[4096];
    const u32 G = m * k, S = G + m;
    const u32 wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const u32 pair = blockIdx.y;
    if (pair < G && pair % k == 0 && blockIdx.x == 0 && wave == 3) {
        const u32 j = pair / k;
        u32 kk;
        const float wt = route_weights(logits + (u64) j * ne, ne, k, lane, (const u32*) pbuf + pair, &kk);
        if (lane < k) ((float*) (pbuf + G * 4))[pair + lane] = wt;
        if (lane == 0) ((u32*) (pbuf + 2 * G * 4))[j] = kk;
    }
    const u8* w;
    if (pair < G) {
        const u32 e = ((const u32*) pbuf)[pair];
        if (e == 0xffffffffu) return;
        w = (const u8*) (ebase + e * estride + 2 * (u64) part);
    } else {
        if (!shbase) return;
        w = (const u8*) (shbase + 2 * (u64) part);
    }
    const float* g = eg + (u64) pair * ff;
    const float* up = eg + (u64) (S + pair) * ff;
    const float* xp[1] = {act};
    float* yp[1] = {eo + (u64) pair * hidden};
    const u32 U = ff / 32;
    if (ff <= 1024 && U <= 64 && 64 % U == 0 && gridDim.x * rpb >= hidden) {
        // one chunk a workgroup and a row's units inside a wave: the launch-1 sums are requested first, the chunk's rows
        // next, and act is made while the rows are on their way (rows_body would take the two round trips in turn)
        const u32 tid = threadIdx.x;
        float gv[4], uv[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const u32 c = min(tid + 256 * i, ff - 1);
            gv[i] = g[c];
            uv[i] = up[c];
        }
        if constexpr (F::BB == 110) {
            for (u32 i = tid; i < 512; i += 256) sz_iq3s_grid[i] = IQ3S_GRID[i];
        }
        const u32 rb = ff / F::QK * F::BB;
        const u32 r0 = blockIdx.x * rpb;
        const u32 head = stage_span(w + (u64) r0 * rb, min(rpb, hidden - r0) * rb, tid);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const u32 c = tid + 256 * i;
            if (c < ff) act[(c / 32) * XU_PITCH + c % 32] = siluf_ref(gv[i]) * uv[i];
        }
        __syncthreads();
        rows_one_chunk<F>(w, hidden, ff, rpb, head, act, yp[0]);
        return;
    }
    for (u32 i = threadIdx.x; i < ff; i += 256) act[i] = siluf_ref(g[i]) * up[i];
    __syncthreads();
    rows_body<F, 1>(w, hidden, ff, rpb, xp, yp, nullptr, NoAfter());
}

// ------------------------------------------------------------------------ the decode layer (one token) in two launches
// For a single token the down launch can own a row chunk for ALL of the token's experts, weight and add them in rank order
// itself, and the combine launch goes away.  Launch 1 then hands over act = silu(gate) * up instead of the two sums (a
// workgroup takes the same rows of gate and of up), and one wave of it computes the routing weights, which launch 2 only reads.
// pbuf as above; act holds S rows of ff floats.  The sums are rows_body's single-input sums and the combine is
// moe_combine_qwen_rows's arithmetic; the routing weights are ex_t over the sum of the chosen ex (route_weights_chosen), within
// a unit in the last place of the three-launch form's, so y agrees with that form to the last bit or two, not bit for bit.

// floor(x / d) for x < 65536 by one multiplication: `magic` = fast_div_magic(d), 1 <= d < 65536 (the one division, done once).
__device__ __forceinline__ u32 fast_div_magic(u32 d) { return 0xffffffffu / d + 1u; }
__device__ __forceinline__ u32 fast_div(u32 x, u32 magic) { return __umulhi(x, magic); }

// Copies `n` spans of `span` bytes into LDS regions of `rs` bytes each (a multiple of 16, at least span + 15): span p starts
// at global address g0(p) and lands so that its first byte is at byte (g0(p) & 15) of region p, which starts at dynamic LDS
// byte p * rs; a null g0(p) skips the span.  All the loads of a thread (at most 4: n * rs / 16 <= 1024) are in flight
// before its first store; a chunk that reaches outside its span is read byte by byte, so nothing outside the spans is touched.
template <class Addr>
__device__ __forceinline__ void stage_spans(Addr g0, u32 n, u32 span, u32 rs, u32 tid) {
    const u32 ch = rs / 16, total = n * ch, nthr = blockDim.x, mch = fast_div_magic(ch);
    u32x4 v[4];
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const u32 i = tid + nthr * r;
        v[r] = u32x4{0, 0, 0, 0};
        if (i < total) {
            const u32 p = fast_div(i, mch), c = i - p * ch;
            const u8* g = g0(p);
            if (g) {
                const u32 head = (u32) ((u64) g & 15);
                const u8* a0 = g - head;
                const u32 lo = c * 16, end = head + span;
                if (lo >= head && lo + 16 <= end) {
                    v[r] = *(const u32x4*) (a0 + lo);
                } else if (lo < end && lo + 16 > head) {
                    u32 w[4] = {0, 0, 0, 0};
                    for (u32 b = 0; b < 16; b++) {
                        const u32 idx = lo + b;
                        if (idx >= head && idx < end) w[b / 4] |= (u32) a0[idx] << (8 * (b % 4));
                    }
                    v[r] = u32x4{w[0], w[1], w[2], w[3]};
                }
            }
        }
    }
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const u32 i = tid + nthr * r;
        if (i < total) ((u32x4*) sz_dyn_lds)[i] = v[r];
    }
}

// Launch 1: as verify_gate_up_gguf for one chunk a workgroup, but the workgroup takes rows [rp blockIdx.x, +rp) of gate AND
// of up and writes act.  The workgroup blockIdx.x == 0 of every token's last pair (the shared expert's, or rank 0's when
// there is none) also selects all k experts on a wave of its own and leaves ids, weights and count in pbuf.
// grid = (ff / rp, S), block 256 to 1024 (a wave takes the rows wave, wave + waves, ..), dynamic LDS = 2 * (rp * row bytes + 32); hidden / 32 divides 64, rp divides ff.
template <class F>
__device__ __forceinline__ void decode_gate_up_gguf(const float* logits, u64 ebase, u64 estride, u64 shbase, u32 part, const float* u, u8* pbuf,
                                                    float* act, u32 ne, u32 k, u32 m, u32 hidden, u32 ff, u32 rp) {
    __shared__ u32 s_top[16], s_all[16];
    __shared__ double s_ex[512], s_ex_all[512];   // only the exact fallback of the routing touches them
    __shared__ __attribute__((aligned(16))) float s_x[64 * XU_PITCH];
    const u32 G = m * k, S = G + m;
    const u32 wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const u32 pair = blockIdx.y;
    const u32 j = pair < G ? pair / k : pair - G;
    if (pair >= G && !shbase) return;
    for (u32 i = threadIdx.x; i < hidden / 4; i += blockDim.x) *(f32x4*) (s_x + (i / 8) * XU_PITCH + (i % 8) * 4) = ((const f32x4*) (u + (u64) j * hidden))[i];
    if constexpr (F::BB == 110) {
        for (u32 i = threadIdx.x; i < 512; i += blockDim.x) sz_iq3s_grid[i] = IQ3S_GRID[i];
    }
    const u32 rwave = (blockIdx.x + blockIdx.y) & 3u;             // the wave that finds this pair's expert
    const bool all = blockIdx.x == 0 && pair == (shbase ? G + j : j * k);
    if (all && wave == ((rwave + 1) & 3u)) {
        const float* lg = logits + (u64) j * ne;
        __builtin_amdgcn_s_setprio(3);
        route_ids(lg, ne, k, lane, s_ex_all, s_all);
        u32 kk;
        const float wt = route_weights_chosen(lg, ne, k, lane, s_all, &kk);
        if (lane < k) {
            ((u32*) pbuf)[j * k + lane] = s_all[lane];
            ((float*) (pbuf + G * 4))[j * k + lane] = wt;
        }
        if (lane == 0) ((u32*) (pbuf + 2 * G * 4))[j] = kk;
        __builtin_amdgcn_s_setprio(0);
    }
    const u8* w;
    if (pair < G) {
        const u32 t = pair % k;
        if (wave == rwave) {
            // the wave every other wave of the workgroup waits for: it goes first where it shares a SIMD with waves of
            // workgroups that are already multiplying
            __builtin_amdgcn_s_setprio(3);
            route_id_of_rank(logits + (u64) j * ne, ne, k, t, lane, s_ex, s_top);   // only s_top[t] is read
            __builtin_amdgcn_s_setprio(0);
        }
        __syncthreads();
        const u32 e = s_top[t];
        if (e == 0xffffffffu) return;
        w = (const u8*) (ebase + e * estride);
    } else {
        w = (const u8*) shbase;
    }
    const u32 rb = hidden / F::QK * F::BB, r0 = blockIdx.x * rp;
    const u32 rs = (rp * rb + 31) / 16 * 16;
    stage_spans([&](u32 p) { return w + (u64) p * part + (u64) r0 * rb; }, 2, rp * rb, rs, threadIdx.x);
    __syncthreads();       // the rows, and for the shared expert's pairs also s_x and the table
    const u32 hg = (u32) ((u64) (w + (u64) r0 * rb) & 15), hu = rs + (u32) ((u64) (w + (u64) part + (u64) r0 * rb) & 15);
    const u32 U = hidden / 32, lg = 31u - (u32) __builtin_clz(U), RG = 64u >> lg, sub = lane >> lg, ul = lane & (U - 1);   // U divides 64: a power of two
    float x[32][1];
    unit_from_lds(s_x, ul, x);
    float* o = act + (u64) pair * ff + r0;
    for (u32 lr = wave * RG + sub; lr < rp; lr += (blockDim.x / 64) * RG) {
        float g[1] = {0.0f}, up[1] = {0.0f};
        unit_dot<F, 1>(hg + lr * rb, ul, x, g);
        unit_dot<F, 1>(hu + lr * rb, ul, x, up);
        g[0] = seg_sum_rt(g[0], U, lane);
        up[0] = seg_sum_rt(up[0], U, lane);
        if (ul == 0) o[lr] = siluf_ref(g[0]) * up[0];
    }
}

// Launch 2 for one token: rows [rd blockIdx.x, +rd) of the down matrix of every chosen expert and of the shared one against
// that pair's act, then y = the sum in rank order of weight * row, plus sigmoid(gate logit) * the shared expert's row.
// grid = hidden / rd, block 256 to 1024 (a wave takes the pairs wave, wave + waves, ..), dynamic LDS = S * region + S * (ff / 32) * 144 with region = rd * row bytes + 31 rounded
// down to 16; ff / 32 divides 64, 64 / (ff / 32) divides rd, rd divides hidden, S * region <= 16 KiB, S * ff <= 8192, k <= 16.
template <class F>
__device__ __forceinline__ void decode_down_combine_gguf(u64 ebase, u64 estride, u64 shbase, u32 part, const u8* pbuf, const float* act,
                                                         const float* gl, float* y, u32 k, u32 hidden, u32 ff, u32 rd) {
    __shared__ float s_eo[17][64];
    __shared__ float s_w[16];
    const u32 G = k, S = shbase ? k + 1 : k;
    const u32 tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const u32 rb = ff / F::QK * F::BB, r0 = blockIdx.x * rd;
    const u32 rs = (rd * rb + 31) / 16 * 16;
    const u32 U = ff / 32, nthr = blockDim.x;
    float* s_act = (float*) ((u8*) sz_dyn_lds + S * rs);
    // every load goes out before anything is waited for: the pairs' act, the chosen ids, then the rows
    const u32 n4 = ff / 4, pieces = S * n4;
    f32x4 av[8];
#pragma unroll
    for (int h = 0; h < 8; h++) av[h] = ((const f32x4*) act)[min(tid + nthr * h, pieces - 1)];
    const u32 myid = ((const u32*) pbuf)[min(lane, k - 1)];
    const float wt = ((const float*) (pbuf + G * 4))[min(lane, k - 1)];
    const u32 cnt = ((const u32*) (pbuf + 2 * G * 4))[0];
    const float glv = shbase ? gl[0] : 0.0f;
    if constexpr (F::BB == 110) {
        for (u32 i = tid; i < 512; i += nthr) sz_iq3s_grid[i] = IQ3S_GRID[i];
    }
    if (wave == 0 && lane < 16) s_w[lane] = lane < k ? wt : 0.0f;
    // the experts' addresses need the ids, which every wave holds in its lanes 0..k-1: a wave-level broadcast
    auto row_of = [&](u32 p) -> const u8* {
        if (p >= G) return (const u8*) (shbase + 2 * (u64) part + (u64) r0 * rb);
        const u32 e = (u32) __shfl((int) myid, (int) p, SZ_WAVE);
        return e == 0xffffffffu ? nullptr : (const u8*) (ebase + e * estride + 2 * (u64) part + (u64) r0 * rb);
    };
    // as stage_spans, with every lane fetching the id of its chunk's pair from the lane that holds it
    {
        const u32 ch = rs / 16, total = S * ch, mch = fast_div_magic(ch), mn4 = fast_div_magic(n4);
        u32x4 v[4];
        const u8* src[4];
        u32 lo[4], hd[4];
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const u32 i = min(tid + nthr * r, total - 1), p = fast_div(i, mch);
            const u8* g = nullptr;
            // (p differs between the lanes of a wave: every lane fetches its pair's id from the lane that holds it)
            if (p >= G) g = (const u8*) (shbase + 2 * (u64) part + (u64) r0 * rb);
            const u32 e = (u32) __shfl((int) myid, (int) min(p, k - 1), SZ_WAVE);
            if (p < G && e != 0xffffffffu) g = (const u8*) (ebase + e * estride + 2 * (u64) part + (u64) r0 * rb);
            src[r] = g;
            hd[r] = (u32) ((u64) g & 15);
            lo[r] = (i - p * ch) * 16;
        }
#pragma unroll
        for (int r = 0; r < 4; r++) {
            v[r] = u32x4{0, 0, 0, 0};
            const u32 i = tid + nthr * r;
            if (i < total && src[r]) {
                const u8* a0 = src[r] - hd[r];
                const u32 end = hd[r] + rd * rb;
                if (lo[r] >= hd[r] && lo[r] + 16 <= end) {
                    v[r] = *(const u32x4*) (a0 + lo[r]);
                } else if (lo[r] < end && lo[r] + 16 > hd[r]) {
                    u32 w[4] = {0, 0, 0, 0};
                    for (u32 b = 0; b < 16; b++) {
                        const u32 idx = lo[r] + b;
                        if (idx >= hd[r] && idx < end) w[b / 4] |= (u32) a0[idx] << (8 * (b % 4));
                    }
                    v[r] = u32x4{w[0], w[1], w[2], w[3]};
                }
            }
        }
#pragma unroll
        for (int h = 0; h < 8; h++) {
            const u32 i = tid + nthr * h;
            if (i < pieces) {
                const u32 p = fast_div(i, mn4), q = i - p * n4;
                *(f32x4*) (s_act + (p * U + q / 8) * XU_PITCH + (q % 8) * 4) = av[h];
            }
        }
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const u32 i = tid + nthr * r;
            if (i < total) ((u32x4*) sz_dyn_lds)[i] = v[r];
        }
    }
    __syncthreads();
    const u32 lg = 31u - (u32) __builtin_clz(U), RG = 64u >> lg, sub = lane >> lg, ul = lane & (U - 1);   // U divides 64: a power of two
    for (u32 p = wave; p < S; p += nthr / 64) {
        const u8* g = row_of(p);
        if (!g) continue;                       // a masked rank: nothing was staged and nothing is added
        const u32 head = p * rs + (u32) ((u64) g & 15);
        float x[32][1];
        unit_from_lds(s_act + p * U * XU_PITCH, ul, x);
        for (u32 lr = sub; lr < rd; lr += RG) {
            float tot[1] = {0.0f};
            unit_dot<F, 1>(head + lr * rb, ul, x, tot);
            tot[0] = seg_sum_rt(tot[0], U, lane);
            if (ul == 0) s_eo[p][lr] = tot[0];
        }
    }
    __syncthreads();
    if (tid < rd) {
        float acc = 0.0f;
        for (u32 t = 0; t < k; t++)
            if (t < cnt) acc += s_w[t] * s_eo[t][tid];
        if (shbase) acc += sigmoidf_ref(glv) * s_eo[G][tid];
        y[r0 + tid] = acc;
    }
}

extern "C" __global__ void __launch_bounds__(1024) decode_gate_up_q8_0(const float* logits, u64 ebase, u64 estride, u64 shbase, u32 part,
                                                                      const float* u, u8* pbuf, float* act, u32 ne, u32 k, u32 m, u32 hidden,
                                                                      u32 ff, u32 rp) {
    decode_gate_up_gguf<Q80>(logits, ebase, estride, shbase, part, u, pbuf, act, ne, k, m, hidden, ff, rp);
}
extern "C" __global__ void __launch_bounds__(1024) decode_gate_up_iq3_s(const float* logits, u64 ebase, u64 estride, u64 shbase, u32 part,
                                                                       const float* u, u8* pbuf, float* act, u32 ne, u32 k, u32 m, u32 hidden,
                                                                       u32 ff, u32 rp) {
    decode_gate_up_gguf<IQ3S>(logits, ebase, estride, shbase, part, u, pbuf, act, ne, k, m, hidden, ff, rp);
}
extern "C" __global__ void __launch_bounds__(1024) decode_down_combine_q8_0(u64 ebase, u64 estride, u64 shbase, u32 part, const u8* pbuf,
                                                                           const float* act, const float* gl, float* y, u32 k, u32 hidden,
                                                                           u32 ff, u32 rd) {
    decode_down_combine_gguf<Q80>(ebase, estride, shbase, part, pbuf, act, gl, y, k, hidden, ff, rd);
}
extern "C" __global__ void __launch_bounds__(1024) decode_down_combine_iq3_s(u64 ebase, u64 estride, u64 shbase, u32 part, const u8* pbuf,
                                                                            const float* act, const float* gl, float* y, u32 k, u32 hidden,
                                                                            u32 ff, u32 rd) {
    decode_down_combine_gguf<IQ3S>(ebase, estride, shbase, part, pbuf, act, gl, y, k, hidden, ff, rd);
}

extern "C" __global__ void __launch_bounds__(256) verify_gate_up_q8_0(const float* logits, u64 ebase, u64 estride, u64 shbase, u32 part,
                                                                      const float* u, u8* pbuf, float* eg, u32 ne, u32 k, u32 m, u32 hidden,
                                                                      u32 ff, u32 rpb) {
    verify_gate_up_gguf<Q80>(logits, ebase, estride, shbase, part, u, pbuf, eg, ne, k, m, hidden, ff, rpb);
}

extern "C" __global__ void __launch_bounds__(256) verify_down_q8_0(const float* logits, u64 ebase, u64 estride, u64 shbase, u32 part, u8* pbuf,
                                                                   const float* eg, float* eo, u32 ne, u32 k, u32 m, u32 hidden, u32 ff,
                                                                   u32 rpb) {
    verify_down_gguf<Q80>(logits, ebase, estride, shbase, part, pbuf, eg, eo, ne, k, m, hidden, ff, rpb);
}

extern "C" __global__ void __launch_bounds__(256) verify_gate_up_iq3_s(const float* logits, u64 ebase, u64 estride, u64 shbase, u32 part,
                                                                      const float* u, u8* pbuf, float* eg, u32 ne, u32 k, u32 m, u32 hidden,
                                                                      u32 ff, u32 rpb) {
    verify_gate_up_gguf<IQ3S>(logits, ebase, estride, shbase, part, u, pbuf, eg, ne, k, m, hidden, ff, rpb);
}

extern "C" __global__ void __launch_bounds__(256) verify_down_iq3_s(const float* logits, u64 ebase, u64 estride, u64 shbase, u32 part, u8* pbuf,
                                                                   const float* eg, float* eo, u32 ne, u32 k, u32 m, u32 hidden, u32 ff,
                                                                   u32 rpb) {
    verify_down_gguf<IQ3S>(logits, ebase, estride, shbase, part, pbuf, eg, eo, ne, k, m, hidden, ff, rpb);
}

// ------------------------------------------------------------------------------- unquantized matrices (F32, F16, BF16)
// The router, the shared expert's gate, the hyper-connection's and other small projections are stored unquantized
// (quant.rs:237-239).  These products are small: what bounds them is the number of memory round trips one after the other,
// so everything a wave needs is requested at once and straight into registers: its share of the inputs (16 columns a lane of
// every row of the batch, kept over all of its rows) and its rows' weights, the next rows' while these are multiplied.
// A row of up to 1024 columns is G lanes' work (64 / G rows a wave at once), a longer one that of several waves of the
// workgroup, whose sums meet in LDS.  Which lane adds which columns, and in which order, depends on the number of columns
// and the type alone: every input of a batch has the bits of a launch of its own.
// cols is a multiple of 4, rows of x are 16-byte aligned, rows of w are aligned to 4 weights, rows >= 1.
typedef u32 u32x4h __attribute__((ext_vector_type(4), aligned(8)));   // 8 two-byte weights, aligned as 4 are
typedef u32 u32x2h __attribute__((ext_vector_type(2), aligned(8)));

struct DenseF32 {
    static constexpr u32 BYTES = 4, C = 4;   // columns a load
    typedef f32x4 Raw;
    static __device__ __forceinline__ Raw load(const u8* p) { return *(const f32x4*) p; }
    static __device__ __forceinline__ Raw none() { return f32x4{0.0f, 0.0f, 0.0f, 0.0f}; }
    static __device__ __forceinline__ float get(const Raw& r, int i) { return r[i]; }
};
template <bool BF, int C_>
struct Dense16 {   // F16, or BF16: the upper half of an f32 (half.rs)
    static constexpr u32 BYTES = 2, C = C_;
    typedef u32 Raw __attribute__((ext_vector_type(C_ / 2)));
    static __device__ __forceinline__ Raw load(const u8* p) {
        if constexpr (C_ == 8) return *(const u32x4h*) p;
        else return *(const u32x2h*) p;
    }
    static __device__ __forceinline__ Raw none() {
        Raw r;
#pragma unroll
        for (int i = 0; i < C_ / 2; i++) r[i] = 0;
        return r;
    }
    static __device__ __forceinline__ float get(const Raw& r, int i) {
        const u32 w = r[i / 2];
        if constexpr (BF) return bits_f32((i & 1) ? w & 0xffff0000u : w << 16);
        else return f16_to_f32((u16) ((i & 1) ? w >> 16 : w));
    }
};

// What a job does to a finished product t: 0 nothing; 1 silu(t / div); 2 2 sigmoid(t / div); 3 sigmoid(t) - the
// hyper-connection's down, inject and up projections (forward.rs:804-814).
__device__ __forceinline__ float dense_act(float t, u32 act, float div) {
    if (act == 1) return siluf_ref(t / div);
    if (act == 2) return 2.0f * sigmoidf_ref(t / div);
    if (act == 3) return sigmoidf_ref(t);
    return t;
}

#define DENSE_LANE_COLS 16u   // columns a lane keeps of every input

// Lanes a row of `cols` columns takes in a wave (a power of two), and waves.
__device__ __forceinline__ u32 dense_lanes(u32 cols) {
    u32 g = 64;
    while (g > 1 && (g / 2) * DENSE_LANE_COLS >= cols) g /= 2;
    return g;
}
__device__ __forceinline__ u32 dense_waves(u32 cols) { return min(8u, (cols + 64 * DENSE_LANE_COLS - 1) / (64 * DENSE_LANE_COLS)); }

// Sums v[j] over the G lanes of a row.  Where G >= M the first log2 M steps halve the number of values a lane carries: lane
// gl then returns output gl % M; else every lane gets every output (v).  The tree of additions is the same for every M.
template <int M>
__device__ __forceinline__ float dense_reduce(float (&v)[M], u32 G, u32 lane) {
    if (G >= (u32) M) {
        if constexpr (M >= 2) {
#pragma unroll
            for (int p = 0; p < M / 2; p++) {
                const bool up = lane & 1;
                v[p] = (up ? v[2 * p + 1] : v[2 * p]) + lane_xor<1>(up ? v[2 * p] : v[2 * p + 1], lane);
            }
        }
        if constexpr (M >= 4) {
#pragma unroll
            for (int p = 0; p < M / 4; p++) {
                const bool up = lane & 2;
                v[p] = (up ? v[2 * p + 1] : v[2 * p]) + lane_xor<2>(up ? v[2 * p] : v[2 * p + 1], lane);
            }
        }
        if constexpr (M >= 8) {
            const bool up = lane & 4;
            v[0] = (up ? v[1] : v[0]) + lane_xor<4>(up ? v[0] : v[1], lane);
        }
        float t = v[0];
        if (M < 2 && G > 1) t += lane_xor<1>(t, lane);
        if (M < 4 && G > 2) t += lane_xor<2>(t, lane);
        if (M < 8 && G > 4) t += lane_xor<4>(t, lane);
        if (G > 8) t += lane_xor<8>(t, lane);
        if (G > 16) t += lane_xor<16>(t, lane);
        if (G > 32) t += lane_xor<32>(t, lane);
        return t;
    }
#pragma unroll
    for (int j = 0; j < M; j++) v[j] = seg_sum_rt(v[j], G, lane);
    return 0.0f;
}

// One lane's columns of a row or of the inputs: chunk i starts at column ((o * NCH + i) * kw_n + kw) * G * C + gl * C.
template <class T>
struct DenseSlice {
    static constexpr int NCH = DENSE_LANE_COLS / T::C;
    u32 kw, kwn, G, gl, cols;
    __device__ __forceinline__ u32 col(u32 o, int i) const { return (((o * NCH + i) * kwn + kw) * G + gl) * T::C; }
    __device__ __forceinline__ void weights(const u8* row, u32 o, bool live, typename T::Raw (&w)[NCH]) const {
#pragma unroll
        for (int i = 0; i < NCH; i++) {
            const u32 c = col(o, i);
            w[i] = T::none();
            if (live && c < cols) w[i] = T::load(row + (u64) c * T::BYTES);
        }
    }
    template <int M>
    __device__ __forceinline__ void inputs(const float* x, u32 xs, u32 m, u32 o, float (&xv)[M][DENSE_LANE_COLS]) const {
#pragma unroll
        for (int j = 0; j < M; j++) {
#pragma unroll
            for (int i = 0; i < NCH; i++) {
                const u32 c = col(o, i);
#pragma unroll
                for (u32 q = 0; q < T::C; q += 4) {
                    f32x4 t = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
                    if ((u32) j < m && c < cols) t = *(const f32x4*) (x + (u64) j * xs + c + q);
#pragma unroll
                    for (int e = 0; e < 4; e++) xv[j][i * T::C + q + e] = t[e];
                }
            }
        }
    }
    template <int M>
    __device__ __forceinline__ void dot(const typename T::Raw (&w)[NCH], const float (&xv)[M][DENSE_LANE_COLS], float (&acc)[M]) const {
#pragma unroll
        for (int i = 0; i < NCH; i++)
#pragma unroll
            for (int e = 0; e < (int) T::C; e++) {
                const float wv = T::get(w[i], e);
#pragma unroll
                for (int j = 0; j < M; j++) acc[j] = __builtin_fmaf(wv, xv[j][i * T::C + e], acc[j]);
            }
    }
};

// Rows [first, first + np * rows a pass) of W against the m inputs by the workgroup (256 threads, or 64 dense_waves(cols) where
// that is more): emit(row, j, sum) once for every output.  red: 2 * 8 * 8 floats of LDS.
template <class T, int M, class Emit>
__device__ __forceinline__ void dense_rows(const u8* __restrict__ w, const float* __restrict__ x, u32 xs, u32 rows, u32 cols, u32 m, u32 first, u32 np,
                                           float* red, Emit emit) {
    typedef DenseSlice<T> S;
    const u32 tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const u32 kwn = dense_waves(cols), G = dense_lanes(cols), rw = (blockDim.x >> 6) / kwn, rg = wave / kwn, per = 64 / G;
    const S sl{wave - rg * kwn, kwn, G, lane & (G - 1), cols};
    const u32 outer = (cols + kwn * G * DENSE_LANE_COLS - 1) / (kwn * G * DENSE_LANE_COLS);
    const bool live = rg < rw;
    u32 row = first + rg * per + lane / G;
    const u32 step = rw * per;
    float xv[M][DENSE_LANE_COLS];
    typename T::Raw wv[S::NCH], wn[S::NCH];
    sl.weights(w + (u64) min(row, rows - 1) * cols * T::BYTES, 0, live && row < rows, wv);
    sl.inputs(x, xs, m, 0, xv);
    for (u32 p = 0; p < np; p++, row += step) {
        const u32 next = row + step;
        const bool more = p + 1 < np;
        if (more) sl.weights(w + (u64) min(next, rows - 1) * cols * T::BYTES, 0, live && next < rows, wn);
        float acc[M];
#pragma unroll
        for (int j = 0; j < M; j++) acc[j] = 0.0f;
        for (u32 o = 0; o < outer; o++) {
            if (outer > 1 && o + p > 0) {   // (rows of more than 8192 columns: the inputs do not stay)
                if (o) sl.weights(w + (u64) min(row, rows - 1) * cols * T::BYTES, o, live && row < rows, wv);
                sl.inputs(x, xs, m, o, xv);
            }
            sl.dot(wv, xv, acc);
        }
        const float t = dense_reduce<M>(acc, G, lane);
        if (kwn == 1) {
            if (live && row < rows) {
                if (G >= (u32) M) {
                    if (sl.gl < m && sl.gl < (u32) M) emit(row, sl.gl, t);
                } else if (sl.gl == 0) {
#pragma unroll
                    for (int j = 0; j < M; j++)
                        if ((u32) j < m) emit(row, (u32) j, acc[j]);
                }
            }
        } else {
            // (a row is at least one whole wave here: G = 64)
            float* r = red + (p & 1) * 64;
            if (live && lane < (u32) M) r[wave * 8 + lane] = t;
            __syncthreads();
            const u32 q = tid / 8, j = tid & 7, orow = first + p * step + q;
            if (q < rw && j < m && orow < rows) {
                float s = r[q * kwn * 8 + j];
                for (u32 v = 1; v < kwn; v++) s += r[(q * kwn + v) * 8 + j];
                emit(orow, j, s);
            }
        }
#pragma unroll
        for (int i = 0; i < S::NCH; i++) wv[i] = wn[i];
    }
}

// The same with the matrix's type picked at run time; two-byte rows that are no multiple of 8 columns are read 4 at a time.
template <int M, class Emit>
__device__ __forceinline__ void dense_rows_of(u32 type, const u8* w, const float* x, u32 xs, u32 rows, u32 cols, u32 m, u32 first, u32 np, float* red, Emit emit) {
    if (type == 0) dense_rows<DenseF32, M>(w, x, xs, rows, cols, m, first, np, red, emit);
    else if (type == 1) {
        if (cols % 8 == 0) dense_rows<Dense16<false, 8>, M>(w, x, xs, rows, cols, m, first, np, red, emit);
        else dense_rows<Dense16<false, 4>, M>(w, x, xs, rows, cols, m, first, np, red, emit);
    } else {
        if (cols % 8 == 0) dense_rows<Dense16<true, 8>, M>(w, x, xs, rows, cols, m, first, np, red, emit);
        else dense_rows<Dense16<true, 4>, M>(w, x, xs, rows, cols, m, first, np, red, emit);
    }
}

// y_j = W x_j for an unquantized row-major W[rows][cols], j < m (matvec_cols_*, kernels/matvec.cu:677): m1, m4 and m8 for
// batches of 1, up to 4 and up to 8, whose inputs take 16, 64 and 128 registers.  type 0 F32, 1 F16, 2 BF16.
// grid = ceil(rows / (np * rows a pass)), block max(256, 64 dense_waves(cols)); a pass is (waves / dense_waves) * 64 / G rows.
template <int M>
__device__ __forceinline__ void dense_cols(u32 type, const u8* w, const float* x, u32 xs, float* y, u32 ys, u32 rows, u32 cols, u32 m, u32 np) {
    __shared__ float red[128];
    const u32 pass = (blockDim.x >> 6) / dense_waves(cols) * (64 / dense_lanes(cols));
    dense_rows_of<M>(type, w, x, xs, rows, cols, m, blockIdx.x * np * pass, np, red, [&](u32 row, u32 j, float t) { y[(u64) j * ys + row] = t; });
}
extern "C" __global__ void __launch_bounds__(512) matvec_cols_dense_m1(u32 type, const u8* w, const float* x, u32 xs, float* y, u32 ys, u32 rows, u32 cols, u32 m, u32 np) {
    dense_cols<1>(type, w, x, xs, y, ys, rows, cols, m, np);
}
extern "C" __global__ void __launch_bounds__(512) matvec_cols_dense_m4(u32 type, const u8* w, const float* x, u32 xs, float* y, u32 ys, u32 rows, u32 cols, u32 m, u32 np) {
    dense_cols<4>(type, w, x, xs, y, ys, rows, cols, m, np);
}
extern "C" __global__ void __launch_bounds__(512) matvec_cols_dense_m8(u32 type, const u8* w, const float* x, u32 xs, float* y, u32 ys, u32 rows, u32 cols, u32 m, u32 np) {
    dense_cols<8>(type, w, x, xs, y, ys, rows, cols, m, np);
}

// The router and the shared expert's gate logit on the same inputs in one launch (moe_router_batch of the reference): the
// router's ne rows into rl[j * ne + row], then, in workgroups of their own, the gate's one row into sgl[j] (gate_w 0: none).
// grid = ceil(ne / pass) (+ 1), block as above, one pass a workgroup.
template <int M>
__device__ __forceinline__ void router_rows(u32 type, const u8* w, u32 gate_type, const u8* gate_w, const float* x, float* rl, float* sgl, u32 ne, u32 cols, u32 m) {
    __shared__ float red[128];
    const u32 pass = (blockDim.x >> 6) / dense_waves(cols) * (64 / dense_lanes(cols)), groups = (ne + pass - 1) / pass;
    if (blockIdx.x < groups) dense_rows_of<M>(type, w, x, cols, ne, cols, m, blockIdx.x * pass, 1, red, [&](u32 row, u32 j, float t) { rl[(u64) j * ne + row] = t; });
    else if (gate_w) dense_rows_of<M>(gate_type, gate_w, x, cols, 1, cols, m, 0, 1, red, [&](u32, u32 j, float t) { sgl[j] = t; });
}
extern "C" __global__ void __launch_bounds__(512) router_rows_m1(u32 type, const u8* w, u32 gate_type, const u8* gate_w, const float* x, float* rl, float* sgl, u32 ne, u32 cols,
                                                                 u32 m) {
    router_rows<1>(type, w, gate_type, gate_w, x, rl, sgl, ne, cols, m);
}
extern "C" __global__ void __launch_bounds__(512) router_rows_m4(u32 type, const u8* w, u32 gate_type, const u8* gate_w, const float* x, float* rl, float* sgl, u32 ne, u32 cols,
                                                                 u32 m) {
    router_rows<4>(type, w, gate_type, gate_w, x, rl, sgl, ne, cols, m);
}
extern "C" __global__ void __launch_bounds__(512) router_rows_m8(u32 type, const u8* w, u32 gate_type, const u8* gate_w, const float* x, float* rl, float* sgl, u32 ne, u32 cols,
                                                                 u32 m) {
    router_rows<8>(type, w, gate_type, gate_w, x, rl, sgl, ne, cols, m);
}

// The hyper-connection's read (forward.rs:797-812) in two launches.  The first: every stream of every row normalised, the mean
// of squares and the scaling of every input in f64 as the CPU path has them, and the down and inject products of that.  A
// workgroup owns `pass` rows of the two matrices (down's first) and normalises the inputs for itself: it has to read all of them
// anyway, and the arithmetic is less than another launch costs.  That arithmetic, in f64, is what bounds it, not the weights: two
// workgroups on a compute unit take nearly twice as long as one.  hc_down_rows_m* take np rows in each group of dense_waves(ch)
// waves, one after the other, the next row's weights on their way, so that one workgroup a unit does (4 rows of 8192 bf16 columns,
// rank 320: 11.9 us -> 9.2); hc_down_m* one row.  Workgroup 0 leaves the scales 1/sqrt(ms + eps) for the second launch.
// r: [m][streams * h]; down, g: silu(t / streams), 2 sigmoid(t / streams).  grid = ceil(rank / pass) + ceil(streams / pass) (inject), np <= HC_NP (1 for hc_down_m*),
// block 64 max(4, dense_waves(ch)), dynamic LDS = m * streams * (1 + chunks of ch) doubles.
__device__ __forceinline__ double lane_xor_f64(double v, u32 lane, int h) {
    const u64 b = __builtin_bit_cast(u64, v);
    float lo = bits_f32((u32) b), hi = bits_f32((u32) (b >> 32));
    switch (h) {
        case 1: lo = lane_xor<1>(lo, lane); hi = lane_xor<1>(hi, lane); break;
        case 2: lo = lane_xor<2>(lo, lane); hi = lane_xor<2>(hi, lane); break;
        case 4: lo = lane_xor<4>(lo, lane); hi = lane_xor<4>(hi, lane); break;
        case 8: lo = lane_xor<8>(lo, lane); hi = lane_xor<8>(hi, lane); break;
        case 16: lo = lane_xor<16>(lo, lane); hi = lane_xor<16>(hi, lane); break;
        default: lo = lane_xor<32>(lo, lane); hi = lane_xor<32>(hi, lane); break;
    }
    return __builtin_bit_cast(double, (u64) f32_bits(lo) | ((u64) f32_bits(hi) << 32));
}
// Sums v[j] over the wave: lane l returns the sum of input l % M (the first log2 M steps halve the number of values a lane carries).
template <int M>
__device__ __forceinline__ double wave_sums_f64(double (&v)[M], u32 lane) {
#pragma unroll
    for (int h = 1; h < M; h *= 2) {
        const bool up = lane & h;
#pragma unroll
        for (int p = 0; p < M / (2 * h); p++) v[p] = (up ? v[2 * p + 1] : v[2 * p]) + lane_xor_f64(up ? v[2 * p] : v[2 * p + 1], lane, h);
    }
    double t = v[0];
#pragma unroll
    for (int h = M; h < 64; h *= 2) t += lane_xor_f64(t, lane, h);
    return t;
}

// The lane's inputs normalised: (float) (r * scale) * norm weight, a chunk of them in one stream.
template <class T, int M>
__device__ __forceinline__ void hc_normalise(const DenseSlice<T>& sl, float (&xv)[M][DENSE_LANE_COLS], const float (&nv)[1][DENSE_LANE_COLS], const double* scl, u32 h, u32 cs, u32 m,
                                             u32 o) {
#pragma unroll
    for (int i = 0; i < DenseSlice<T>::NCH; i++) {
        const u32 s = min(sl.col(o, i), sl.cols - 1) / h;
#pragma unroll
        for (int j = 0; j < M; j++) {
            if ((u32) j < m) {
                const double sc = scl[(u32) j * cs + s];
#pragma unroll
                for (int e = 0; e < (int) T::C; e++) xv[j][i * T::C + e] = (float) ((double) xv[j][i * T::C + e] * sc) * nv[0][i * T::C + e];
            }
        }
    }
}

#define HC_NP 4u   // rows of a wave at most
template <class T, int M, bool MANY>
__device__ __forceinline__ void hc_down_rows(const u8* __restrict__ w, u32 rows, u32 first, const float* __restrict__ r, const float* __restrict__ nw, double* __restrict__ scales,
                                             u32 h, u32 cs, u32 m, float eps, u32 np, float* red, u32 act, float* y, u32 ys) {
    typedef DenseSlice<T> S;
    if constexpr (!MANY) np = 1;
    const u32 tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const u32 cols = h * cs, kwn = dense_waves(cols), rw = (blockDim.x >> 6) / kwn, rg = wave / kwn;
    const S sl{wave - rg * kwn, kwn, 64, lane, cols};
    const u32 span = 64 * T::C, outer = (cols + kwn * span * S::NCH - 1) / (kwn * span * S::NCH);
    double* part = (double*) sz_dyn_lds;       // [m][cs][spans of 64 C columns a stream can touch]: their sums of squares, a span one wave's, in order
    const u32 wide = h / span + 2;
    double* scl = part + (u64) m * cs * wide;
    const bool live = rg < rw;
    auto weights = [&](u32 q, u32 o, typename T::Raw (&raw)[S::NCH]) {   // of the wave's q-th row
        const u32 row = first + q * rw + rg;
        sl.weights(w + (u64) min(row, rows - 1) * cols * T::BYTES, o, live && o < outer && row < rows, raw);
    };
    float xv[M][DENSE_LANE_COLS];
    typename T::Raw wv[S::NCH], wn[S::NCH];
    weights(0, 0, wv);
    sl.inputs(r, cols, m, 0, xv);
    for (u32 i = tid; i < m * cs * wide; i += blockDim.x) part[i] = 0.0;
    __syncthreads();
    // the spans' sums of squares first, then the products (of inputs that are still in registers where outer == 1)
    for (u32 o = 0; o < outer; o++) {
        if (o) sl.inputs(r, cols, m, o, xv);
#pragma unroll
        for (int i = 0; i < S::NCH; i++) {
            const u32 c0 = ((o * S::NCH + i) * kwn + sl.kw) * span;   // the span's first column: a span touches one stream, or several where h is small
            const u32 c = c0 + lane * T::C, mine = c / h;
            if (rg == 0 && c0 < cols) {
                double sq[M];
#pragma unroll
                for (int j = 0; j < M; j++) {
                    sq[j] = 0.0;
                    if (c < cols)
#pragma unroll
                        for (int e = 0; e < (int) T::C; e++) sq[j] = __builtin_fma((double) xv[j][i * T::C + e], (double) xv[j][i * T::C + e], sq[j]);
                }
                for (u32 s = c0 / h; s <= (min(c0 + span, cols) - 1) / h; s++) {
                    double of[M];
#pragma unroll
                    for (int j = 0; j < M; j++) of[j] = mine == s ? sq[j] : 0.0;
                    const double ss = wave_sums_f64<M>(of, lane);
                    if (lane < (u32) M && lane < m) part[((u64) lane * cs + s) * wide + (c0 / span - s * h / span)] = ss;
                }
            }
        }
    }
    float nv[1][DENSE_LANE_COLS];   // the norm weights come while the scales are made
    sl.inputs(nw, 0, 1, 0, nv);
    u32 qn = 0, on = 0;   // the row and the columns that wn is of
    auto next = [&]() {
        if (++qn == np) qn = 0, on++;
        weights(qn, on, wn);
    };
    if constexpr (MANY) next();
    __syncthreads();
    for (u32 i = tid; i < m * cs; i += blockDim.x) {
        double ss = 0.0;
        for (u32 q = 0; q < wide; q++) ss += part[i * wide + q];
        const double sc = 1.0 / sqrt(ss / (double) h + (double) eps);
        scl[i] = sc;
        if (blockIdx.x == 0) scales[i] = sc;
    }
    __syncthreads();
    if constexpr (MANY) {
        float acc[HC_NP][M];   // a lane's own over all its columns, as below: a row's bits are the same in either form
#pragma unroll
        for (int q = 0; q < (int) HC_NP; q++)
#pragma unroll
            for (int j = 0; j < M; j++) acc[q][j] = 0.0f;
        for (u32 o = 0; o < outer; o++) {
            if (outer > 1) {
                sl.inputs(r, cols, m, o, xv);
                sl.inputs(nw, 0, 1, o, nv);
            }
            hc_normalise<T, M>(sl, xv, nv, scl, h, cs, m, o);
#pragma unroll
            for (u32 q = 0; q < HC_NP; q++) {
                if (q >= np) break;
                sl.dot(wv, xv, acc[q]);
#pragma unroll
                for (int i = 0; i < S::NCH; i++) wv[i] = wn[i];
                next();
                if (o + 1 < outer) continue;
                const float t = dense_reduce<M>(acc[q], 64, lane);
                if (live && lane < (u32) M) red[(q * 8 + wave) * 8 + lane] = t;
            }
        }
    } else {
        float acc[M];
#pragma unroll
        for (int j = 0; j < M; j++) acc[j] = 0.0f;
        for (u32 o = 0; o < outer; o++) {
            if (outer > 1) {
                weights(0, o, wv);
                sl.inputs(r, cols, m, o, xv);
                sl.inputs(nw, 0, 1, o, nv);
            }
            hc_normalise<T, M>(sl, xv, nv, scl, h, cs, m, o);
            sl.dot(wv, xv, acc);
        }
        const float t = dense_reduce<M>(acc, 64, lane);
        if (live && lane < (u32) M) red[wave * 8 + lane] = t;
    }
    __syncthreads();
    const u32 orow = tid / 8, j = tid & 7, q = orow / rw, og = orow - q * rw;
    if (q < np && j < m && first + orow < rows) {
        const float* part8 = red + (q * 8 + og * kwn) * 8 + j;
        float s = part8[0];
        for (u32 v = 1; v < kwn; v++) s += part8[v * 8];
        y[(u64) j * ys + first + orow] = dense_act(s, act, (float) cs);
    }
}
template <int M, bool MANY>
__device__ __forceinline__ void hc_down_of(u32 type, const u8* w, u32 rows, u32 first, const float* r, const float* nw, double* scales, u32 h, u32 cs, u32 m, float eps, u32 np, float* red,
                                           u32 act, float* y, u32 ys) {
    // spans stay whole inside a stream's 4-column groups: 8 columns a load only where a stream is a multiple of 8
    if (type == 0) hc_down_rows<DenseF32, M, MANY>(w, rows, first, r, nw, scales, h, cs, m, eps, np, red, act, y, ys);
    else if (type == 1) {
        if (h % 8 == 0) hc_down_rows<Dense16<false, 8>, M, MANY>(w, rows, first, r, nw, scales, h, cs, m, eps, np, red, act, y, ys);
        else hc_down_rows<Dense16<false, 4>, M, MANY>(w, rows, first, r, nw, scales, h, cs, m, eps, np, red, act, y, ys);
    } else {
        if (h % 8 == 0) hc_down_rows<Dense16<true, 8>, M, MANY>(w, rows, first, r, nw, scales, h, cs, m, eps, np, red, act, y, ys);
        else hc_down_rows<Dense16<true, 4>, M, MANY>(w, rows, first, r, nw, scales, h, cs, m, eps, np, red, act, y, ys);
    }
}
template <int M, bool MANY>
__device__ __forceinline__ void hc_down(u32 type, const u8* w, u32 rank, u32 gate_type, const u8* gate_w, const float* r, const float* nw, u8* scales, float* down, float* g, u32 h,
                                        u32 cs, u32 m, float eps, u32 np) {
    __shared__ float red[(MANY ? HC_NP : 1) * 64];
    if constexpr (!MANY) np = 1;
    const u32 pass = (blockDim.x >> 6) / dense_waves(h * cs) * np, groups = (rank + pass - 1) / pass;
    if (blockIdx.x < groups) hc_down_of<M, MANY>(type, w, rank, blockIdx.x * pass, r, nw, (double*) scales, h, cs, m, eps, np, red, 1, down, rank);
    else hc_down_of<M, MANY>(gate_type, gate_w, cs, (blockIdx.x - groups) * pass, r, nw, (double*) scales, h, cs, m, eps, np, red, 2, g, cs);
}
extern "C" __global__ void __launch_bounds__(512) hc_down_m1(u32 type, const u8* w, u32 rank, u32 gate_type, const u8* gate_w, const float* r, const float* nw, u8* scales, float* down,
                                                             float* g, u32 h, u32 cs, u32 m, float eps, u32 np) {
    hc_down<1, false>(type, w, rank, gate_type, gate_w, r, nw, scales, down, g, h, cs, m, eps, np);
}
extern "C" __global__ void __launch_bounds__(512, 4) hc_down_m4(u32 type, const u8* w, u32 rank, u32 gate_type, const u8* gate_w, const float* r, const float* nw, u8* scales, float* down,
                                                             float* g, u32 h, u32 cs, u32 m, float eps, u32 np) {
    hc_down<4, false>(type, w, rank, gate_type, gate_w, r, nw, scales, down, g, h, cs, m, eps, np);
}
extern "C" __global__ void __launch_bounds__(512) hc_down_m8(u32 type, const u8* w, u32 rank, u32 gate_type, const u8* gate_w, const float* r, const float* nw, u8* scales, float* down,
                                                             float* g, u32 h, u32 cs, u32 m, float eps, u32 np) {
    hc_down<8, false>(type, w, rank, gate_type, gate_w, r, nw, scales, down, g, h, cs, m, eps, np);
}
extern "C" __global__ void __launch_bounds__(512) hc_down_rows_m1(u32 type, const u8* w, u32 rank, u32 gate_type, const u8* gate_w, const float* r, const float* nw, u8* scales, float* down,
                                                             float* g, u32 h, u32 cs, u32 m, float eps, u32 np) {
    hc_down<1, true>(type, w, rank, gate_type, gate_w, r, nw, scales, down, g, h, cs, m, eps, np);
}
extern "C" __global__ void __launch_bounds__(512) hc_down_rows_m4(u32 type, const u8* w, u32 rank, u32 gate_type, const u8* gate_w, const float* r, const float* nw, u8* scales, float* down,
                                                             float* g, u32 h, u32 cs, u32 m, float eps, u32 np) {
    hc_down<4, true>(type, w, rank, gate_type, gate_w, r, nw, scales, down, g, h, cs, m, eps, np);
}
extern "C" __global__ void __launch_bounds__(512) hc_down_rows_m8(u32 type, const u8* w, u32 rank, u32 gate_type, const u8* gate_w, const float* r, const float* nw, u8* scales, float* down,
                                                             float* g, u32 h, u32 cs, u32 m, float eps, u32 np) {
    hc_down<8, true>(type, w, rank, gate_type, gate_w, r, nw, scales, down, g, h, cs, m, eps, np);
}

// The second: u[j][i] = (sum over the streams s, in order, of sigmoid(up row s h + i . down_j) * the normalised r[j][s h + i]) / streams.
// A wave takes 64 / G columns i at a time and the streams' rows of them one after the other, the next row's weights and terms on their
// way, so that the sum over the streams needs nobody else.  grid = ceil(h / (4 * 64 / G)), block 256.
template <class T, int M>
__device__ __forceinline__ void hc_up_rows(const u8* __restrict__ w, const float* __restrict__ down, const float* __restrict__ r, const float* __restrict__ nw,
                                           const double* __restrict__ scales, float* __restrict__ u, u32 h, u32 cs, u32 rank, u32 m) {
    typedef DenseSlice<T> S;
    const u32 lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const u32 G = dense_lanes(rank), per = 64 / G;
    const S sl{0, 1, G, lane & (G - 1), rank};
    const u32 i0 = (blockIdx.x * 4 + wave) * per + lane / G, i = min(i0, h - 1);
    const u32 outer = (rank + G * DENSE_LANE_COLS - 1) / (G * DENSE_LANE_COLS);
    // the lane that ends up with output j holds its terms too
    const bool spread = G >= (u32) M;
    const u32 j0 = spread ? min(sl.gl & (M - 1), m - 1) : 0;
    float xv[M][DENSE_LANE_COLS];
    typename T::Raw wv[S::NCH], wn[S::NCH];
    sl.weights(w + (u64) i * rank * T::BYTES, 0, true, wv);
    sl.inputs(down, rank, m, 0, xv);
    float a[M];
#pragma unroll
    for (int j = 0; j < M; j++) a[j] = 0.0f;
    float nn = nw[i], rn = r[(u64) j0 * cs * h + i];
    double scn = scales[j0 * cs];
    for (u32 s = 0; s < cs; s++) {
        const u64 at = (u64) s * h + i;
        const float n = nn, rv = rn;
        const double sc = scn;
        if (s + 1 < cs) {
            sl.weights(w + (at + h) * rank * T::BYTES, 0, true, wn);
            nn = nw[at + h];
            rn = r[(u64) j0 * cs * h + at + h];
            scn = scales[j0 * cs + s + 1];
        }
        float acc[M];
#pragma unroll
        for (int j = 0; j < M; j++) acc[j] = 0.0f;
        for (u32 o = 0; o < outer; o++) {
            if (outer > 1 && o + s > 0) {
                if (o) sl.weights(w + at * rank * T::BYTES, o, true, wv);
                sl.inputs(down, rank, m, o, xv);
            }
            sl.dot(wv, xv, acc);
        }
        const float t = dense_reduce<M>(acc, G, lane);
        if (spread) {
            a[0] += sigmoidf_ref(t) * ((float) ((double) rv * sc) * n);
        } else {
#pragma unroll
            for (int j = 0; j < M; j++)
                if ((u32) j < m) a[j] += sigmoidf_ref(acc[j]) * ((float) ((double) r[(u64) j * cs * h + at] * scales[j * cs + s]) * n);
        }
#pragma unroll
        for (int q = 0; q < S::NCH; q++) wv[q] = wn[q];
    }
    if (i0 < h) {
        if (spread) {
            if (sl.gl < m && sl.gl < (u32) M) u[(u64) sl.gl * h + i] = a[0] / (float) cs;
        } else if (sl.gl == 0) {
#pragma unroll
            for (int j = 0; j < M; j++)
                if ((u32) j < m) u[(u64) j * h + i] = a[j] / (float) cs;
        }
    }
}
template <int M>
__device__ __forceinline__ void hc_up(u32 type, const u8* w, const float* down, const float* r, const float* nw, const u8* scales, float* u, u32 h, u32 cs, u32 rank, u32 m) {
    const double* sc = (const double*) scales;
    if (type == 0) hc_up_rows<DenseF32, M>(w, down, r, nw, sc, u, h, cs, rank, m);
    else if (type == 1) {
        if (rank % 8 == 0) hc_up_rows<Dense16<false, 8>, M>(w, down, r, nw, sc, u, h, cs, rank, m);
        else hc_up_rows<Dense16<false, 4>, M>(w, down, r, nw, sc, u, h, cs, rank, m);
    } else {
        if (rank % 8 == 0) hc_up_rows<Dense16<true, 8>, M>(w, down, r, nw, sc, u, h, cs, rank, m);
        else hc_up_rows<Dense16<true, 4>, M>(w, down, r, nw, sc, u, h, cs, rank, m);
    }
}
extern "C" __global__ void __launch_bounds__(256) hc_up_m1(u32 type, const u8* w, const float* down, const float* r, const float* nw, const u8* scales, float* u, u32 h, u32 cs,
                                                           u32 rank, u32 m) {
    hc_up<1>(type, w, down, r, nw, scales, u, h, cs, rank, m);
}
extern "C" __global__ void __launch_bounds__(256) hc_up_m4(u32 type, const u8* w, const float* down, const float* r, const float* nw, const u8* scales, float* u, u32 h, u32 cs,
                                                           u32 rank, u32 m) {
    hc_up<4>(type, w, down, r, nw, scales, u, h, cs, rank, m);
}
extern "C" __global__ void __launch_bounds__(256) hc_up_m8(u32 type, const u8* w, const float* down, const float* r, const float* nw, const u8* scales, float* u, u32 h, u32 cs,
                                                           u32 rank, u32 m) {
    hc_up<8>(type, w, down, r, nw, scales, u, h, cs, rank, m);
}

// ------------------------------------------------------------------------------------------------ lm_head + argmax
// The head product for m <= 4 rows with each workgroup's (maximum, lowest index) of every row over all its row chunks
// written to part[(blockIdx.x * 4 + j) * 2] = {value bits, index}, so the logits never have to be written (logits may be
// null).  A NaN logit counts as -inf, as the device top-k does (kernels/forward.cu:3592).  grid = any number of workgroups up
// to the number of chunks, block 256, dynamic LDS = rpb * row bytes + 32 + rpb * 16.
extern "C" __global__ void __launch_bounds__(256) head_q8_0_argmax(const u8* w, const float* x, u32 xs, float* logits, u32 ls, u32* part,
                                                                   u32 rows, u32 cols, u32 m, u32 rpb) {
    const u32 n = min(4u, m);
    const u32 rb = cols / 32 * 34;
    float* res = (float*) (sz_dyn_lds + (rpb * rb + 32 + 3) / 4);
    const float* xp[4];
    float* yp[4];
    for (u32 j = 0; j < 4; j++) {
        const u32 jj = j < n ? j : 0;
        xp[j] = x + (u64) jj * xs;
        yp[j] = (j < n && logits) ? logits + (u64) jj * ls : nullptr;
    }
    float bv = -__builtin_inff();
    u32 bi = 0xffffffffu;
    const u32 tid = threadIdx.x;
    auto after = [&](u32 r0, u32 nrows) {
        if (tid < n) {
            for (u32 r = 0; r < nrows; r++) {
                float v = res[r * 4 + tid];
                if (v != v) v = -__builtin_inff();
                argmax_merge(bv, bi, v, r0 + r);
            }
        }
    };
    rows_dispatch<Q80>(w, rows, cols, rpb, n, xp, yp, res, after);
    if (tid < n) {
        part[((u64) blockIdx.x * 4 + tid) * 2] = f32_bits(bv);
        part[((u64) blockIdx.x * 4 + tid) * 2 + 1] = bi;
    }
}

// The same head on the matrix cores, for W = 4, 6 or 8 waves and cols <= 512 W (a multiple of 64 W), m <= 8 and a 16-byte aligned matrix.
// A 16-row tile of the matrix (16 x cols / 32 x 34 contiguous bytes) comes into LDS by global-to-LDS loads, the next tile
// while this one is multiplied.  Wave w owns the share k in [w cols / W, (w + 1) cols / W) of every row and keeps its
// slice of the inputs in registers for the whole launch, as the B operands of v_mfma_f32_16x16x16_f16: with
// s_j x_j = the input row times the power of two that takes its largest magnitude to [2^14, 2^15), column 2 j holds
// f16(s_j x_j) and column 2 j + 1 holds f16(s_j x_j - f16(s_j x_j)): the high parts are finite whatever the activations'
// size, the two columns together carry an element to 22 bits unless it is below 2^-17 of the row's largest (there the
// low part runs into f16's subnormals and the element keeps at least its 11 high-part bits, an error below 2^-39 of
// the largest), and every product with the int8 codes (exact in f16) is exact; the matrix core adds in f32 and the sums
// are multiplied by 1 / s_j at the end.  The A operand is the tile's
// codes: a lane takes 4 consecutive codes of row lane % 16, turns each into the f16 1024 + (code ^ 0x80) by putting 0x64
// above the byte, and subtracts 1152 (exact).  A 32-block's two products are scaled by the block's f16 scale and added to
// the lane's running sums in f32, block after block in k order; the waves' sums are added in wave order.
// part[(blockIdx.x * 8 + j) * 2] = {value bits, index} of the workgroup's best row for input j (NaN counts as -inf,
// ties to the lower index).  grid <= tiles (persistent: tile t goes to workgroup t % grid), block 64 W.
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
#define HEAD_PITCH(cols) ((cols) / 32 * 34 + 16)   // bytes between a tile's rows in LDS: 16 rows then fall on different banks

__device__ __forceinline__ f16x4 head_codes_f16(u32 q) {
    const u32 u = q ^ 0x80808080u;                                   // code + 128 as unsigned bytes
    const u32 lo = __builtin_amdgcn_perm(0x64646464u, u, 0x04010400u);   // halves 0x6400 | byte 0, 0x6400 | byte 1
    const u32 hi = __builtin_amdgcn_perm(0x64646464u, u, 0x04030402u);
    typedef _Float16 f16x2_ __attribute__((ext_vector_type(2)));
    const f16x2_ k = {(_Float16) -1152.0f, (_Float16) -1152.0f};
    const f16x2_ a = __builtin_bit_cast(f16x2_, lo) + k, b = __builtin_bit_cast(f16x2_, hi) + k;
    return f16x4{a[0], a[1], b[0], b[1]};
}

// Requests tile `t` (rows 16 t .. 16 t + 15, clamped to the last row) into the LDS buffer at byte offset `lds`: wave w of W
// brings rows w, w + W, .., each as 16-byte pieces (ceil(row bytes / 1024) instructions a row).  once: past the caches.
template <int W, bool once>
__device__ __forceinline__ void head_tile_rows(const u8* __restrict__ w, u32 rows, u32 rb, u32 t, u32 lds, u32 wave, u32 lane) {
    const u32 pieces = rb / 16;                           // rb is a multiple of 16 here
#pragma unroll
    for (int rr = 0; rr < (16 + W - 1) / W; rr++) {
        const u32 lr = wave + W * rr;
        if (lr < 16) {
            const u8* src = w + (u64) min(16 * t + lr, rows - 1) * rb;
            const u32 dst = lds + lr * (rb + 16);
#pragma unroll
            for (int c = 0; c < 5; c++)
                if (c * 64 < pieces)
                    if (c * 64 + lane < pieces) lds_load<16, once>(src + (c * 64 + lane) * 16, dst + c * 1024);
        }
    }
}
// A head of 256 MiB or more, what the last level holds, goes past the caches, out of which it would push everything else (the 64 best of 4
// rows of 151 936 x 2048, 315 MiB, 107 us, 98.7; of 8 of 65 536 x 4096, 272 MiB, 121, 117.5; a round of 2 layers with the first 96, 90, of 4 with
// four rows 134, 132).  A smaller one is there again at the next call, also with layers in between (4 rows of 151 936 x 1024, 158 MiB, 86 and past
// the caches 91; rounds of 1 to 16 layers with 65 536 x 2560, 170 MiB, 85, 104, 129, 173, 257 and 88, 108, 135, 178, 262; with 249 MiB 0 to 2 %
// apart).  The choice stands outside the loops: at every load it cost those heads 1 to 2 %.
template <int W>
__device__ __forceinline__ void head_tile_issue(const u8* __restrict__ w, u32 rows, u32 rb, u32 t, u32 lds, u32 wave, u32 lane) {
    if ((u64) rows * rb >= 256u << 20) head_tile_rows<W, true>(w, rows, rb, t, lds, wave, lane);
    else head_tile_rows<W, false>(w, rows, rb, t, lds, wave, lane);
}

// W waves (4, 6 or 8), cols = CMAX (512 W unless a narrower row is given more waves) at most and a multiple of 64 W.
template <int W, int CMAX = 512 * W, bool FULL = false>   // FULL: cols == CMAX, every wave owns NBM blocks (no per-block checks: the tile reads of all blocks go out together)
__device__ __forceinline__ void head_mfma_body(const u8* w, const float* x, u32 xs, float* logits, u32 ls, u32* part, u32 rows, u32 cols, u32 m) {
    __shared__ float s_bv[256];
    __shared__ u32 s_bi[256];
    __shared__ float s_mx[W][8], s_inv[8];   // largest magnitude of a wave's share of every input row; the factor that undoes a row's scale
    const u32 tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    if constexpr (FULL) cols = CMAX;                      // (the host launches this form for no other width: offsets become constants)
    const u32 rb = cols / 32 * 34, pitch = rb + 16;
    constexpr int NBM = CMAX / W / 32;                    // the most 32-blocks a wave owns
    const u32 kw = cols / W, nbw = kw / 32;               // a wave's columns, and their 32-blocks (<= NBM)
    const u32 n16 = lane & 15, g4 = lane >> 4;
    __shared__ __attribute__((aligned(16))) u8 tiles_lds[2 * 16 * HEAD_PITCH(CMAX)];   // two tiles, 16 * pitch bytes apart
    __shared__ float red[W][256];
    u8* const tile0 = tiles_lds;
    // the wave's slice of the inputs as B operands: B[k = 4 g4 + i][n = n16], n = 2 j + (0: high part, 1: low part)
    f16x4 xb[NBM][2];
    {
        const u32 j = n16 >> 1, lowpart = n16 & 1;
        // all 32 loads go out before the first is waited for (clamped to an address that exists where the lane has no
        // input or the block lies past the row: a load behind a branch is waited for on the spot, a round trip each)
        f32x4 raw[NBM][2];
        const float* xj = x + (u64) min(j, m - 1) * xs + wave * kw + 4 * g4;
#pragma unroll
        for (int b = 0; b < NBM; b++)
#pragma unroll
            for (int h = 0; h < 2; h++) raw[b][h] = *(const f32x4*) (xj + 32 * min((u32) b, nbw - 1) + 16 * h);
        // every input row is scaled by a power of two that takes its largest magnitude to [2^14, 2^15) before it is split (the
        // sums are scaled back at the end): the high parts cannot overflow to infinity whatever the activations' size, and
        // the low parts of small activations are not lost to f16's subnormal range
        float mxl = 0.0f;
#pragma unroll
        for (int b = 0; b < NBM; b++)
#pragma unroll
            for (int h = 0; h < 2; h++)
                if (FULL || (u32) b < nbw)
#pragma unroll
                    for (int i = 0; i < 4; i++) mxl = fmaxf(mxl, __builtin_fabsf(raw[b][h][i]));   // a NaN is skipped here and shows in the sums
        mxl = fmaxf(mxl, lane_xor<16>(mxl, lane));
        mxl = fmaxf(mxl, lane_xor<32>(mxl, lane));
        if (g4 == 0 && lowpart == 0) s_mx[wave][j] = mxl;
        __syncthreads();
        float mxr = s_mx[0][j];
#pragma unroll
        for (int v = 1; v < W; v++) mxr = fmaxf(mxr, s_mx[v][j]);
        float scale, inv;
        pow2_scale_of(f32_bits(mxr), scale, inv);
        if (wave == 0 && g4 == 0 && lowpart == 0) s_inv[j] = inv;
#pragma unroll
        for (int b = 0; b < NBM; b++)
#pragma unroll
            for (int h = 0; h < 2; h++) {
                f16x4 v = {0, 0, 0, 0};
                if ((FULL || (u32) b < nbw) && j < m) {
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const float f = raw[b][h][i] * scale;
                        const _Float16 hi = (_Float16) f;
                        v[i] = lowpart ? (_Float16) (f - (float) hi) : hi;
                    }
                }
                xb[b][h] = v;
                asm volatile("" : "+v"(xb[b][h]));   // consumed here: no ordinary load of the inputs is in flight once the tiles are requested
            }
    }
    const u32 tiles = (rows + 15) / 16;
    const u32 lds0 = __builtin_amdgcn_readfirstlane(lds_offset(tile0)), lds1 = lds0 + 16 * pitch;
    // the load instructions a tile costs this wave: its rows (w, w + W, .. < 16) times the 1 KiB pieces of a row
    const u32 mine = ((16 - wave + W - 1) / W) * ((rb / 16 + 63) / 64);
    float bv = -__builtin_inff();
    u32 bi = 0xffffffffu;
    u32 t = blockIdx.x, it = 0;
    if (t < tiles) head_tile_issue<W>(w, rows, rb, t, lds0, wave, lane);
    for (; t < tiles; t += gridDim.x, it++) {
        const u32 tn = t + gridDim.x;
        if (tn < tiles) head_tile_issue<W>(w, rows, rb, tn, (it & 1) ? lds0 : lds1, wave, lane);
        // this tile's requests of this wave have landed; the next tile's (the youngest in the queue) may stay in flight -
        // unless logits are stored in the loop: a store is not ordered with the loads
        if (tn < tiles && !logits) {
            if (mine >= 12) wait_vm<12>();
            else if (mine >= 10) wait_vm<10>();
            else if (mine >= 8) wait_vm<8>();
            else if (mine >= 4) wait_vm<4>();
            else wait_vm<0>();
        } else {
            wait_vm<0>();
        }
        __syncthreads();                                  // ... and every other wave's
        const u8* tb = tile0 + (it & 1) * 16 * pitch;
        const u8* arow = tb + n16 * pitch + wave * nbw * 34;      // A: row n16 of the tile, the wave's share of k
        const u8* drow = tb + (4 * g4) * pitch + wave * nbw * 34;  // scales: rows 4 g4 + r
        float tot[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int b = 0; b < NBM; b++) {
            if (FULL || (u32) b < nbw) {
                const u8* ab = arow + b * 34 + 2 + 4 * g4;
                const u32 q0 = *(const u16*) ab | ((u32) *(const u16*) (ab + 2) << 16);
                const u32 q1 = *(const u16*) (ab + 16) | ((u32) *(const u16*) (ab + 18) << 16);
                f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
                acc = __builtin_amdgcn_mfma_f32_16x16x16f16(head_codes_f16(q0), xb[b][0], acc, 0, 0, 0);
                acc = __builtin_amdgcn_mfma_f32_16x16x16f16(head_codes_f16(q1), xb[b][1], acc, 0, 0, 0);
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const _Float16 d = __builtin_bit_cast(_Float16, *(const u16*) (drow + r * pitch + b * 34));
                    tot[r] = __builtin_fmaf((float) d, acc[r], tot[r]);
                }
            }
        }
#pragma unroll
        for (int r = 0; r < 4; r++) red[wave][(4 * g4 + r) * 16 + n16] = tot[r];
        __syncthreads();
        if (tid < 256) {
            // thread (row = tid / 16, n = tid % 16): the waves' sums in wave order, then high part + low part
            float s = red[0][tid];
#pragma unroll
            for (int v = 1; v < W; v++) s += red[v][tid];
            const float o = lane_xor<1>(s, lane);
            const u32 n = tid & 15, j = n >> 1, row = 16 * t + (tid >> 4);
            if ((n & 1) == 0 && j < m && row < rows) {
                float v = (s + o) * s_inv[j];
                if (logits) logits[(u64) j * ls + row] = v;
                if (v != v) v = -__builtin_inff();
                argmax_merge(bv, bi, v, row);
            }
        }
    }
    // the workgroup's best row per input: thread (row slot tid / 16, n) holds the best of its row slot
    if (tid < 256) {
        s_bv[tid] = bv;
        s_bi[tid] = bi;
    }
    __syncthreads();
    if (tid < 8) {
        float v = -__builtin_inff();
        u32 i = 0xffffffffu;
        for (u32 r = 0; r < 16; r++) argmax_merge(v, i, s_bv[r * 16 + 2 * tid], s_bi[r * 16 + 2 * tid]);
        part[((u64) blockIdx.x * 8 + tid) * 2] = f32_bits(v);
        part[((u64) blockIdx.x * 8 + tid) * 2 + 1] = i;
    }
}

extern "C" __global__ void __launch_bounds__(256, 2) head_q8_0_argmax_mfma(const u8* w, const float* x, u32 xs, float* logits, u32 ls, u32* part,
                                                                           u32 rows, u32 cols, u32 m) {
    head_mfma_body<4>(w, x, xs, logits, ls, part, rows, cols, m);
}
// The same for rows of up to 3072 columns (6 waves, block 384) and up to 4096 (8 waves, block 512): a wave still owns at
// most 512 columns, the tiles take all of a CU's LDS but for a workgroup's share, so one workgroup a CU.
// Rows of exactly 2048 columns on 8 waves: the same LDS a workgroup, twice the waves a SIMD to cover the tile reads' latency.
extern "C" __global__ void __launch_bounds__(512, 2) head_q8_0_argmax_mfma_n8(const u8* w, const float* x, u32 xs, float* logits, u32 ls, u32* part,
                                                                              u32 rows, u32 cols, u32 m) {
    head_mfma_body<8, 2048, true>(w, x, xs, logits, ls, part, rows, cols, m);
}
extern "C" __global__ void __launch_bounds__(384) head_q8_0_argmax_mfma_w6(const u8* w, const float* x, u32 xs, float* logits, u32 ls, u32* part,
                                                                           u32 rows, u32 cols, u32 m) {
    head_mfma_body<6>(w, x, xs, logits, ls, part, rows, cols, m);
}
extern "C" __global__ void __launch_bounds__(512) head_q8_0_argmax_mfma_w8(const u8* w, const float* x, u32 xs, float* logits, u32 ls, u32* part,
                                                                           u32 rows, u32 cols, u32 m) {
    head_mfma_body<8>(w, x, xs, logits, ls, part, rows, cols, m);
}

// part[(p * ts + j) * 2], + 1 = the largest of slice p (4096 values) of row j of logits (rows ls apart, n values a row) and its
// index, ties to the lower index: the first step of the arg-max for a head whose product kernel has none fused in (any type
// matvec_cols takes; the reference's mv_cols + topk_rows_at, session.rs:7034-7052).  grid = (ceil(n / 4096), m), block 256.
extern "C" __global__ void __launch_bounds__(256) argmax_slices(const float* logits, u32 ls, u32 n, u32* part, u32 ts) {
    __shared__ float sv[256];
    __shared__ u32 si[256];
    const u32 p = blockIdx.x, j = blockIdx.y, tid = threadIdx.x;
    const float* row = logits + (u64) j * ls;
    float bv = -__builtin_inff();
    u32 bi = 0xffffffffu;
#pragma unroll 4
    for (u32 q = 0; q < 16; q++) {
        const u32 i = p * 4096 + q * 256 + tid;
        if (i < n) argmax_merge(bv, bi, row[i], i);
    }
    sv[tid] = bv;
    si[tid] = bi;
    __syncthreads();
    for (u32 s = 128; s > 0; s >>= 1) {
        if (tid < s) {
            float v = sv[tid];
            u32 i = si[tid];
            argmax_merge(v, i, sv[tid + s], si[tid + s]);
            sv[tid] = v;
            si[tid] = i;
        }
        __syncthreads();
    }
    if (tid == 0) {
        part[((u64) p * ts + j) * 2] = f32_bits(sv[0]);
        part[((u64) p * ts + j) * 2 + 1] = si[0];
    }
}

// argmax_merge_parts for all m <= 8 rows and the greedy acceptance in one launch (the end of a verify round: one launch and
// its boundary less): ids[j] as there, then out[0] = keep = 1 + the number of leading drafts d[i] that equal ids[i], out[1] =
// the bonus token ids[keep - 1] (verify_accept in kernels/moe.hip; engine.rs:2377-2408).  grid 1, block 1024 (128 threads a row).
extern "C" __global__ void __launch_bounds__(1024) argmax_merge_accept(const u32* part, u32 nparts, u32 ts, u32* ids, u32 m, const u32* drafts,
                                                                       u32 n_drafts, u32* out) {
    __shared__ float sv[8][128];
    __shared__ u32 si[8][128];
    const u32 j = threadIdx.x >> 7, t = threadIdx.x & 127;
    float bv = -__builtin_inff();
    u32 bi = 0xffffffffu;
    if (j < m)
        for (u32 p = t; p < nparts; p += 128) argmax_merge(bv, bi, bits_f32(part[((u64) p * ts + j) * 2]), part[((u64) p * ts + j) * 2 + 1]);
    sv[j][t] = bv;
    si[j][t] = bi;
    __syncthreads();
    for (u32 s = 64; s > 0; s >>= 1) {
        if (t < s) {
            float v = sv[j][t];
            u32 i = si[j][t];
            argmax_merge(v, i, sv[j][t + s], si[j][t + s]);
            sv[j][t] = v;
            si[j][t] = i;
        }
        __syncthreads();
    }
    if (threadIdx.x < 64) {
        const u32 i = threadIdx.x;
        if (i < m) ids[i] = si[i][0];
        const u32 a = si[min(min(i, n_drafts), 7u)][0];
        const u32 d = i < n_drafts ? drafts[i] : 0u;
        const u64 stop = __builtin_amdgcn_ballot_w64(i >= n_drafts || a != d);
        const u32 first = (u32) __builtin_ctzll(stop);
        const u32 bonus = __builtin_amdgcn_readlane(a, first);
        if (i == 0) {
            out[0] = first + 1;
            out[1] = bonus;
        }
    }
}

// ids[j] = index of the largest of row j's `nparts` partial maxima part[(p * ts + j) * 2] (ties to the lower index).
// grid = m, block 256.
extern "C" __global__ void __launch_bounds__(256) argmax_merge_parts(const u32* part, u32 nparts, u32 ts, u32* ids, float* vals) {
    __shared__ float sv[256];
    __shared__ u32 si[256];
    const u32 j = blockIdx.x, tid = threadIdx.x;
    float bv = -__builtin_inff();
    u32 bi = 0xffffffffu;
    for (u32 p = tid; p < nparts; p += 256) {
        argmax_merge(bv, bi, bits_f32(part[((u64) p * ts + j) * 2]), part[((u64) p * ts + j) * 2 + 1]);
    }
    sv[tid] = bv;
    si[tid] = bi;
    __syncthreads();
    for (u32 s = 128; s > 0; s >>= 1) {
        if (tid < s) {
            float v = sv[tid];
            u32 i = si[tid];
            argmax_merge(v, i, sv[tid + s], si[tid + s]);
            sv[tid] = v;
            si[tid] = i;
        }
        __syncthreads();
    }
    if (tid == 0) {
        ids[j] = si[0];
        if (vals) vals[j] = sv[0];
    }
}
