// k_nnls_lh's own source (cut out of kvc_kernels.hip by the test that builds
// this) on the CPU: every lane is a coroutine, a wave's lanes meet at each
// cross-lane operation, and the waves of the block meet at __syncthreads
// only. Between two block barriers the scheduler runs one wave as far as it
// goes before the other starts, in the order the test names, so a value that
// passes between the waves without a barrier is read stale or overwritten
// every time. LDS arrays are statics, which the undefined-behaviour
// sanitizer bounds and aligns.
//
// stdin: int32 waves, first wave to run, n, max_iter; n (n + 1) floats
// [AtA | Atb]. stdout: n floats; the status word and the redo flag as int32.
#include <ucontext.h>

#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <algorithm>
#include <utility>
#include <vector>

namespace {

using std::min;
using std::max;

struct Dim { unsigned x, y, z; };
struct alignas(16) float4 { float x, y, z, w; };
float4 make_float4(float x, float y, float z, float w) { return {x, y, z, w}; }
struct Geom { int H, n_chunks, t_total; };
struct ChunkDesc { int tc, off; };

enum Meet { NONE, WAVE, BLOCK };
struct Lane {
    Dim tid;
    ucontext_t ctx;
    std::vector<char> stack;
    Meet at = NONE;
    bool done = false;
    unsigned ops = 0;   // cross-lane operations so far
};
std::vector<Lane> lanes;
Lane * cur;
ucontext_t sched;
Dim blockIdx;
unsigned posted[2][2][64];   // [wave][parity of the operation][lane]

void meet(Meet m) {
    cur->at = m;
    swapcontext(&cur->ctx, &sched);
}
// every lane's value of this operation (a lane is at most one operation ahead)
const unsigned * gather(unsigned v) {
    unsigned * p = posted[cur->tid.x >> 6][cur->ops++ & 1];
    p[cur->tid.x & 63] = v;
    meet(WAVE);
    return p;
}

int __float_as_int(float f) { int i; memcpy(&i, &f, 4); return i; }
unsigned __float_as_uint(float f) { unsigned i; memcpy(&i, &f, 4); return i; }
float __int_as_float(int i) { float f; memcpy(&f, &i, 4); return f; }
float __uint_as_float(unsigned i) { float f; memcpy(&f, &i, 4); return f; }
int __popcll(unsigned long long v) { return __builtin_popcountll(v); }
int lane_read(int v, int l) { return (int)gather((unsigned)v)[l & 63]; }
unsigned long long __ballot(bool b) {
    const unsigned * p = gather(b);
    unsigned long long m = 0;
    for (int l = 0; l < 64; l++) m |= (unsigned long long)p[l] << l;
    return m;
}
template <bool MAX>
unsigned dpp_reduce_u32(unsigned v) {
    const unsigned * p = gather(v);
    return MAX ? *std::max_element(p, p + 64) : *std::min_element(p, p + 64);
}
template <int L>
float sb_bc(float v) { return __uint_as_float(gather(__float_as_uint(v))[((cur->tid.x & 63) & ~15u) + L]); }
unsigned score_key(float x) {
    const unsigned b = __float_as_uint(x);
    return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}
void atomicOr(int * p, int v) { *p |= v; }
void wave_meet() { meet(WAVE); }
void __syncthreads() { meet(BLOCK); }

#define __device__
#define __global__
#define __forceinline__ inline
#define __shared__ static
#define __align__(n) __attribute__((aligned(n)))
#define __launch_bounds__(n)
#define amdgpu_waves_per_eu(n) unused
#define threadIdx (cur->tid)
#define __builtin_amdgcn_readlane(v, l) lane_read(v, l)
#define __builtin_amdgcn_readfirstlane(v) lane_read(v, 0)
#define __builtin_amdgcn_fence(order, scope)
#define __builtin_amdgcn_wave_barrier() wave_meet()

#include "lawson_hanson.inc"

Geom geom;
ChunkDesc chunk;
long long aug_off = 0;
std::vector<float> aug, wout;
int max_iter, status = 0, redo = 1, W;

void body() {
    if (W == 1) k_nnls_lh<1>(geom, &chunk, aug.data(), &aug_off, wout.data(), max_iter, &status, &redo);
    else k_nnls_lh<2>(geom, &chunk, aug.data(), &aug_off, wout.data(), max_iter, &status, nullptr);
    cur->done = true;
    swapcontext(&cur->ctx, &sched);
}

// wave w to its next block barrier or its end; false: its lanes diverged
bool run_wave(int w) {
    for (;;) {
        int at[3] = {0, 0, 0}, done = 0;
        for (int l = 0; l < 64; l++) {
            Lane & x = lanes[64 * w + l];
            cur = &x;
            x.at = NONE;
            swapcontext(&sched, &x.ctx);
            done += x.done;
            at[x.at]++;
        }
        if (done == 64 || at[BLOCK] == 64) return true;
        if (at[WAVE] != 64) return false;
    }
}

}  // namespace

int main() {
    int h[4];
    if (fread(h, 4, 4, stdin) != 4) return 2;
    W = h[0];
    const int first = h[1], n = h[2];
    max_iter = h[3];
    if (W < 1 || W > 2 || n < 1 || n > 256) return 2;
    geom = {1, 1, n};
    chunk = {n, 0};
    aug.resize((size_t)n * (n + 1));
    wout.assign(n, 0.0f);
    if (fread(aug.data(), 4, aug.size(), stdin) != aug.size()) return 2;
    lanes.resize(64 * W);
    for (unsigned t = 0; t < lanes.size(); t++) {
        Lane & x = lanes[t];
        x.tid = {t, 0, 0};
        x.stack.resize(256 << 10);
        getcontext(&x.ctx);
        x.ctx.uc_stack.ss_sp = x.stack.data();
        x.ctx.uc_stack.ss_size = x.stack.size();
        makecontext(&x.ctx, body, 0);
    }
    for (;;) {
        int ended = 0;
        for (int k = 0; k < W; k++) {
            const int w = (first + k) % W;
            if (!run_wave(w)) {
                fprintf(stderr, "wave %d: lanes at different operations\n", w);
                return 3;
            }
            ended += lanes[64 * w].done;
        }
        if (ended == W) break;
        if (ended) {
            fprintf(stderr, "one wave ended, the other waits at a barrier\n");
            return 4;
        }
    }
    fwrite(wout.data(), 4, n, stdout);
    const int tail[2] = {status, redo};
    fwrite(tail, 4, 2, stdout);
    return 0;
}
