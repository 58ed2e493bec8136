// The selective-scan branch of a step that brings one row per sequence, in two launches (vx_scan_step): what vx_conv_silu, the split
// map of its result, the map to the channels' time steps and vx_selective_scan compute in five, with the same sums in the same order.
//
// Each of the five is a launch's fixed time and a trip or two to memory (3.8 - 8 us), and a few megabytes at most. What lets them join is that
// a decode step's rows are few enough to be computed again by every workgroup that reads them:
//  * conv_project_kernel: a row tile of the split map and a slice of its inputs, as linear_few_kernel; a lane's operand, eight channels of a
//    row, is convolved in its registers instead of loaded. (Ten row tiles convolve the same channels, 8 K outputs a workgroup: about 1 us.)
//  * scan_project (scan_step.h): 32 channels of 16 rows. The waves add up the slices of the rows' low-rank part as a matrix operand and
//    multiply, add up B and C and move the convolution's history; then two lanes a channel and row step the states, which were asked for
//    at the start.
// 32 rows, 4096 channels x 16 states, rank 128, in a traced step, us: the five launches 5.0 + 4.6 + 3.7 + 4.2 + 7.7, these two 6.6 + 9.2; the second one with
// single-token attention (9.5 - 10 alone) beside it 12.7. (A workgroup of two row tiles convolved twice as much: 9.1.) The step of a bfloat16 model of four such layers with its logits 585 -> 520 - 531.
#include <string.h>

#include "scan_step.h"

using namespace vx;
using namespace vx::scan_step;

namespace {

// Eight channels' convolution of a row from their inputs, the taps' weights and the bias.
__device__ __forceinline__ bf16x8 convolved(const bf16x8 (&v)[TAPS], const f32x8 (&w)[TAPS], f32x8 acc, int pos) {
#pragma unroll
    for (int t = 0; t < TAPS; t++) {
        const bool there = TAPS - 1 - t <= pos;  // (before the sequence's start: zero, whatever an earlier owner left)
#pragma unroll
        for (int e = 0; e < 8; e++) acc[e] = fmaf(w[t][e], there ? (float)v[t][e] : 0.f, acc[e]);
    }
    bf16x8 o;
#pragma unroll
    for (int e = 0; e < 8; e++) o[e] = (bf16)silu_f(acc[e]);
    return o;
}

__global__ void __launch_bounds__(64 * PW, 2) conv_project_kernel(StepArgs a) {
    __shared__ f32x4 red[PW][64];
    const vx_conv_args &p = a.p.conv;
    const int lane = threadIdx.x & 63, wave = wave_id();
    const int steps = a.p.x_k >> 5, slices = gridDim.y, slice = blockIdx.y, tile = blockIdx.x;
    const int s0 = (int)((int64_t)steps * slice / slices), s1 = (int)((int64_t)steps * (slice + 1) / slices);
    const bf16 *w = (const bf16 *)a.p.x_w + (size_t)tile * steps * 512 + lane * 8;
    const int own = blockIdx.z * 16 + (lane & 15), row = min(own, a.rows - 1), pos = a.pos[row];
    const bf16 *x = (const bf16 *)p.x + (size_t)row * p.ldx, *st = (const bf16 *)p.state + (size_t)a.slots[row] * (TAPS - 1) * p.channels;
    f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
    // (everything that two steps read is asked for ahead of the first sum: a wave has up to four steps, and a trip to memory for each was half
    // of the launch)
    constexpr int U = 2;
    for (int sb = s0 + wave; sb < s1; sb += U * PW) {
        bf16x8 wf[U], v[U][TAPS];
        f32x8 cw[U][TAPS], cb[U];
        int c[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int s = min(sb + u * PW, s1 - 1);
            wf[u] = __builtin_nontemporal_load((const bf16x8 *)(w + (size_t)s * 512));
            c[u] = s * 32 + (lane >> 4) * 8;
            const int cc = min(c[u], p.channels - 8);
            cb[u] = *(const f32x8 *)(p.b + cc);
#pragma unroll
            for (int t = 0; t < TAPS; t++) cw[u][t] = *(const f32x8 *)(p.w + (size_t)t * p.channels + cc);
            v[u][TAPS - 1] = *(const bf16x8 *)(x + cc);
#pragma unroll
            for (int t = 0; t + 1 < TAPS; t++) v[u][t] = *(const bf16x8 *)(st + (size_t)t * p.channels + cc);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < U; u++) {
            if (sb + u * PW >= s1) break;
            bf16x8 o = convolved(v[u], cw[u], cb[u], pos);
            if (c[u] >= p.channels)  // (columns that pad the inputs)
#pragma unroll
                for (int e = 0; e < 8; e++) o[e] = (bf16)0.f;
            if (tile == 0 && own < a.rows) *(bf16x8 *)((bf16 *)p.out + (size_t)own * p.ldo + c[u]) = o;
            acc = mma(wf[u], o, acc);
        }
    }
    red[wave][lane] = acc;
    __syncthreads();
    if (wave == 0 && own < a.rows) {
        f32x4 v = red[0][lane];
#pragma unroll
        for (int k = 1; k < PW; k++) v += red[k][lane];
        *(f32x4 *)(a.part + ((size_t)slice * a.rows + own) * a.p.x_n + tile * 16 + (lane >> 4) * 4) = v;
    }
}

__global__ void __launch_bounds__(THREADS, 2) scan_project_kernel(StepArgs a) { scan_project(a, blockIdx.x, blockIdx.y); }

}  // namespace

extern "C" {

// Where the split map is one that vx_linear cuts into slices for linear_few_kernel. (Longer slices would have more of the convolution computed by every row tile:
// those are the maps that linear_hold_kernel takes from 17 rows on.)
int vx_scan_step_takes(vx_backend *be, int act, const vx_ragged *b, const vx_scan_step_args *p) {
    if (!b || !p || act != VX_ACT_BF16 || b->q_lens || b->rows < 1 || b->rows > 64) return 0;
    const vx_conv_args &c = p->conv;
    const vx_scan_args &s = p->scan;
    if (c.taps != TAPS || s.states < 1 || vx_scan_state_pad(s.states) != PAD || c.channels != s.channels || c.channels < 8 || c.channels % 8 != 0) return 0;
    if (p->x_k < 2048 || p->x_k % 64 != 0 || p->x_n % 16 != 0 || p->dt_k < 64 || p->dt_k % 64 != 0 || p->dt_n % 16 != 0 || p->x_n < p->dt_k + 2 * PAD ||
        c.ldo < p->x_k || p->x_k < c.channels || p->dt_n < c.channels)
        return 0;
    const int slices = vx_linear_slices(be, p->x_n, p->x_k, b->rows);
    if (slices < 2 || slices > SLICES || ceil_div(ceil_div(p->x_k >> 5, slices), PW) > 4) return 0;
    const auto al = [](const void *q, int n) { return q && (uintptr_t)q % n == 0; };
    return c.ldx % 8 == 0 && c.ldo % 8 == 0 && c.ldx >= c.channels && al(c.x, 16) && al(c.out, 16) && al(c.state, 16) && al(c.w, 32) && al(c.b, 32) &&
           al(p->x_w, 16) && al(p->dt_w, 16) && p->dt_bias && al(s.a2, 16) && al(s.state, 16) && s.d && s.z && s.out && s.x == c.out && s.ldx == c.ldo &&
           s.ldz >= s.channels && s.out_cols >= s.channels && s.ldo >= s.out_cols;
}

int vx_scan_step(vx_backend *be, int act, const vx_ragged *b, const vx_scan_step_args *p, const vx_attn_args *attn) {
    int rc = enter(be);
    if (rc) return rc;
    rc = check_ragged(b, "vx_scan_step");
    if (rc) return rc;
    VX_REQUIRE(vx_scan_step_takes(be, act, b, p), "vx_scan_step: not for these sizes (vx_scan_step_takes)");
    StepArgs a;
    memset(&a, 0, sizeof a);
    a.p = *p, a.pos = b->token_pos, a.slots = b->table_rows, a.rows = b->rows;
    a.slices = vx_linear_slices(be, p->x_n, p->x_k, b->rows);
    rc = ensure_ws(be, &be->part_ws, &be->part_ws_bytes, (size_t)a.slices * b->rows * p->x_n * 4, "partial sums");
    if (rc) return rc;
    a.part = (float *)be->part_ws;
    conv_project_kernel<<<dim3(p->x_n >> 4, a.slices, ceil_div(b->rows, ROWS)), 64 * PW, 0, be->stream>>>(a);
    VX_CHECK_LAUNCH();
    bool beside = false;
    if (attn) {
        rc = attn_beside(be, act, b, attn, a, &beside);
        if (rc || beside) return rc;
    }
    scan_project_kernel<<<dim3(ceil_div(p->scan.channels, CH), ceil_div(b->rows, ROWS)), THREADS, 0, be->stream>>>(a);
    VX_CHECK_LAUNCH();
    return VX_OK;
}

}  // extern "C"
