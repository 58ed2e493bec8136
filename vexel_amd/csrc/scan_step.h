// The second half of vx_scan_step, as a device function: a launch of its own (scan_step.hip), or workgroups beside those of single-token
// attention (attn_ragged.hip).
#pragma once

#include "ragged.h"

namespace vx {

struct StepArgs {
    vx_scan_step_args p;
    const int32_t *pos, *slots;
    int rows, slices;
    float *part;  // [slices][rows][x_n]
};

namespace scan_step {

constexpr int TAPS = 4, PAD = 16, LP = 2, NS = PAD / LP;  // taps; states of a channel as they are kept, its lanes, states of a lane
constexpr int PW = 8;                                     // waves that share a map's inputs (linear_few_kernel's)
constexpr int CH = 32, ROWS = 16, THREADS = 256;          // channels, rows and threads of a workgroup
constexpr int SLICES = 8;

// N neighbouring pieces of four columns of n <= SLICES slices, asked for in one trip.
template <int N> struct Sliced {
    f32x4 v[SLICES][N];
    __device__ __forceinline__ void ask(const float *at, size_t stride, int n) {
#pragma unroll
        for (int s = 0; s < SLICES; s++)
#pragma unroll
            for (int i = 0; i < N; i++) v[s][i] = *(const f32x4 *)(at + (size_t)min(s, n - 1) * stride + 4 * i);
    }
    __device__ __forceinline__ f32x4 sum(int i, int n) const {  // in their order
        f32x4 y = v[0][i];
#pragma unroll
        for (int s = 1; s < SLICES; s++)
            if (s < n) y += v[s][i];
        return y;
    }
};

__device__ __forceinline__ f32x8 load8(const float *p) {
    const f32x4 a = *(const f32x4 *)p, b = *(const f32x4 *)(p + 4);
    return f32x8{a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
}

// Channels bx * CH .. of rows by * ROWS ...
__device__ __forceinline__ void scan_project(const StepArgs &a, int bx, int by) {
    __shared__ f32x4 red[PW][CH / 16][64];
    __shared__ f32x4 s_bc[ROWS][2 * PAD / 4];
    const vx_scan_args &p = a.p.scan;
    constexpr int WAVES = THREADS / 64, ITEMS = ROWS / WAVES, PER = 2 * PAD / 4;
    static_assert(PW == 2 * WAVES && CH * LP == 64 && ROWS * PER + ROWS * CH / 8 <= THREADS, "who does what");
    const int tid = threadIdx.x, lane = tid & 63, wave = wave_id();
    const int c0 = bx * CH, r0 = by * ROWS;
    const int steps = a.p.dt_k >> 5, n = a.p.x_n, tiles = a.p.dt_n >> 4;
    const size_t stride = (size_t)a.rows * n;
    const int sub = lane & 1, ch = lane >> 1, c = min(c0 + ch, p.channels - 1);
    // what one trip brings: the wave's first step of the rows' low-rank part and of the map, B and C, the states
    const float *src = a.part + (size_t)min(r0 + (lane & 15), a.rows - 1) * n + (lane >> 4) * 8;
    int slot[ITEMS], pos[ITEMS];
#pragma unroll
    for (int i = 0; i < ITEMS; i++) {
        const int row = min(r0 + wave + WAVES * i, a.rows - 1);
        slot[i] = a.slots[row], pos[i] = a.pos[row];
    }
    Sliced<2> low;
    low.ask(src + min(wave, steps - 1) * 32, stride, a.slices);
    Sliced<1> bc;
    if (tid < ROWS * PER) bc.ask(a.part + (size_t)min(r0 + tid / PER, a.rows - 1) * n + a.p.dt_k + tid % PER * 4, stride, a.slices);
    const f32x8 A = load8(p.a2 + (size_t)c * PAD + sub * NS);
    const float D = p.d[c], bias = a.p.dt_bias[c];
    f32x8 S[ITEMS];
    float *state[ITEMS], x[ITEMS], z[ITEMS];
#pragma unroll
    for (int i = 0; i < ITEMS; i++) {
        const int row = min(r0 + wave + WAVES * i, a.rows - 1);
        state[i] = p.state + ((size_t)slot[i] * p.channels + c) * PAD + sub * NS;
        S[i] = load8(state[i]);
        x[i] = (float)((const bf16 *)p.x)[(size_t)row * p.ldx + c];
        z[i] = (float)((const bf16 *)p.z)[(size_t)row * p.ldz + c];
    }
    // this wave's steps and those of the wave WAVES on, in sums of their own
#pragma unroll
    for (int h = 0; h < 2; h++) {
        const int v = wave + h * WAVES;
        f32x4 acc[CH / 16];
#pragma unroll
        for (int t = 0; t < CH / 16; t++) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
        for (int s = v; s < steps; s += PW) {
            bf16x8 wf[CH / 16], u;
#pragma unroll
            for (int t = 0; t < CH / 16; t++)
                wf[t] = *(const bf16x8 *)((const bf16 *)a.p.dt_w + ((size_t)min((c0 >> 4) + t, tiles - 1) * steps + s) * 512 + lane * 8);
            if (s != wave) low.ask(src + s * 32, stride, a.slices);
#pragma unroll
            for (int i = 0; i < 2; i++) {
                const f32x4 y = low.sum(i, a.slices);
#pragma unroll
                for (int e = 0; e < 4; e++) u[i * 4 + e] = (bf16)y[e];
            }
#pragma unroll
            for (int t = 0; t < CH / 16; t++) acc[t] = mma(wf[t], u, acc[t]);
        }
#pragma unroll
        for (int t = 0; t < CH / 16; t++) red[v][t][lane] = acc[t];
    }
    if (tid < ROWS * PER) {
        s_bc[tid / PER][tid % PER] = bc.sum(0, a.slices);
    } else {
        // the convolution's history: entry k is the input of TAPS - 1 - k tokens before the next one
        const vx_conv_args &q = a.p.conv;
        const int j = tid - ROWS * PER, row = r0 + j / (CH / 8), hc = c0 + j % (CH / 8) * 8;
        if (j < ROWS * CH / 8 && row < a.rows && hc < q.channels) {
            bf16 *st = (bf16 *)q.state + (size_t)a.slots[row] * (TAPS - 1) * q.channels + hc;
            const int at = a.pos[row];
            bf16x8 v[TAPS - 1];
#pragma unroll
            for (int k = 0; k + 2 < TAPS; k++) v[k] = *(const bf16x8 *)(st + (size_t)(k + 1) * q.channels);
            v[TAPS - 2] = *(const bf16x8 *)((const bf16 *)q.x + (size_t)row * q.ldx + hc);
#pragma unroll
            for (int k = 0; k + 1 < TAPS; k++) {
                if (at < TAPS - 2 - k)
#pragma unroll
                    for (int e = 0; e < 8; e++) v[k][e] = (bf16)0.f;
                *(bf16x8 *)(st + (size_t)k * q.channels) = v[k];
            }
        }
    }
    __syncthreads();
    const int parts = min(steps, PW);
#pragma unroll
    for (int i = 0; i < ITEMS; i++) {
        const int row = wave + WAVES * i;  // of the tile
        const float *y0 = (const float *)&red[0][ch >> 4][row + 16 * ((ch & 15) >> 2)] + (ch & 3);
        float y = y0[0];
        for (int k = 1; k < parts; k++) y += y0[k * (CH / 16) * 64 * 4];
        const float dt = softplus_f(y + bias), dx = dt * x[i];
        const f32x8 B = load8((const float *)s_bc[row] + sub * NS), C = load8((const float *)s_bc[row] + PAD + sub * NS);
        float o = 0.f;
#pragma unroll
        for (int k = 0; k < NS; k++) S[i][k] = fmaf(__builtin_amdgcn_exp2f(dt * A[k]), pos[i] > 0 ? S[i][k] : 0.f, dx * B[k]);
#pragma unroll
        for (int k = 0; k < NS; k++) o = fmaf(S[i][k], C[k], o);
        o += __shfl_xor(o, 1, 64);
        if (r0 + row >= a.rows || c0 + ch >= p.channels) continue;
        if (sub == 0) ((bf16 *)p.out)[(size_t)(r0 + row) * p.ldo + c] = (bf16)(p.out_scale * (fmaf(D, x[i], o) * silu_f(z[i])));
        *(f32x4 *)state[i] = f32x4{S[i][0], S[i][1], S[i][2], S[i][3]};
        *(f32x4 *)(state[i] + 4) = f32x4{S[i][4], S[i][5], S[i][6], S[i][7]};
    }
    if (bx == 0) {  // the columns that pad the row
        const int w = p.out_cols - p.channels, live = min(ROWS, a.rows - r0);
        for (int i = tid; i < w * live; i += THREADS) ((bf16 *)p.out)[(size_t)(r0 + i / w) * p.ldo + p.channels + i % w] = (bf16)0.f;
    }
}

}  // namespace scan_step

// vx_attn_ragged with such workgroups in its launch, where that is the one of single-token attention on heads of 97 to 128: *beside says
// whether it was. (There it takes registers for two workgroups a compute unit either way; narrower heads have more.)
int attn_beside(vx_backend *be, int act, const vx_ragged *b, const vx_attn_args *p, const StepArgs &scan, bool *beside);

}  // namespace vx
