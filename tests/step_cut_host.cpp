// step_plan.h and step_cut.h compiled for the host: the functions the decode step's launch and its
// kernel run, with a wave's 64 lanes as 64 contexts that take turns at every wave-wide operation
// (control flow around those is uniform, so each lane's turn ends at the same one).
#include <algorithm>
#include <csetjmp>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <ucontext.h>
#include <vector>

#define __device__
#define __forceinline__ inline

namespace lanes {

constexpr int kLanes = 64;
constexpr size_t kStack = 64 << 10;
uint32_t slot[2][kLanes];  // values of the current and the previous operation
int turn[kLanes], lane;
bool done[kLanes], started[kLanes];
jmp_buf at[kLanes], home;
ucontext_t entry[kLanes], main_context;
std::vector<char> stacks(kLanes *kStack);
void (*body)(int);

void enter() {
    body(lane);
    done[lane] = true;
    _longjmp(home, 1);
}
void switch_to(int l) {
    lane = l;
    if (started[l])
        _longjmp(at[l], 1);
    started[l] = true;
    getcontext(&entry[l]);
    entry[l].uc_stack.ss_sp = stacks.data() + l * kStack;
    entry[l].uc_stack.ss_size = kStack;
    entry[l].uc_link = nullptr;
    makecontext(&entry[l], enter, 0);
    setcontext(&entry[l]);
}
// Hands in the lane's value and returns the wave's values once every lane has.
const uint32_t *gather(uint32_t v) {
    const int me = lane;
    uint32_t *s = slot[turn[me]++ & 1];
    s[me] = v;
    if (_setjmp(at[me]) == 0)
        _longjmp(home, 1);
    return s;
}
void run(void (*f)(int)) {
    body = f;
    std::memset(turn, 0, sizeof turn);
    std::memset(done, 0, sizeof done);
    std::memset(started, 0, sizeof started);
    for (static int l; ; ) {
        for (l = 0; l < kLanes; ++l)
            if (!done[l] && _setjmp(home) == 0)
                switch_to(l);
        if (std::all_of(done, done + kLanes, [](bool d) { return d; }))
            return;
    }
}

}  // namespace lanes

namespace tq4 {
namespace xdl {

constexpr int kWave = lanes::kLanes;
template <typename T> T max(T a, T b) { return a > b ? a : b; }
template <typename T> T min(T a, T b) { return a < b ? a : b; }
inline int div_pos(int a, int b) { return a / b; }
inline uint32_t wave_scan(uint32_t v) {
    const uint32_t *s = lanes::gather(v);
    uint32_t sum = 0;
    for (int i = 0; i <= lanes::lane; ++i)
        sum += s[i];
    return sum;
}
inline uint32_t wave_max(uint32_t v) {
    const uint32_t *s = lanes::gather(v);
    return *std::max_element(s, s + kWave);
}
inline uint64_t ballot(bool v) {
    const uint32_t *s = lanes::gather(v);
    uint64_t m = 0;
    for (int i = 0; i < kWave; ++i)
        m |= (uint64_t)(s[i] & 1) << i;
    return m;
}
inline int readlane(int v, int l) { return (int)lanes::gather((uint32_t)v)[l & 63]; }

}  // namespace xdl
}  // namespace tq4

#define __ballot(v) ballot(v)
#define __builtin_amdgcn_readlane(v, l) readlane(v, l)
#define __builtin_amdgcn_readfirstlane(v) readlane(v, 0)
#include "../turboquant-cuda-decode_amd/csrc/step_cut.h"

namespace {

tq4::xdl::CutArgs args;
int nx, x;
tq4::xdl::Cut cuts[lanes::kLanes];
bool found[lanes::kLanes], single[lanes::kLanes];

void one_lane(int lane) {
    tq4::xdl::Cut c{};
    const int len = args.seq_lens[lane < args.batch ? lane : args.batch - 1];
    bool one = true;
    found[lane] = tq4::xdl::first_segment(c, args, nx, x, lane, len, one);
    cuts[lane] = c;
    single[lane] = one;
}

}  // namespace

extern "C" {

// out: vw, sw, nx, per_seq, whole, rotates
void host_step_plan(int held, int nvh, int batch, int max_blocks, int block_size, int num_splits, int whole_lines,
                    int have_parts, int *out) {
    const auto p = tq4::xdl::step_plan(
        {held, nvh, batch, max_blocks, block_size, num_splits, whole_lines != 0}, have_parts != 0);
    out[0] = p.vw, out[1] = p.sw, out[2] = p.nx, out[3] = p.per_seq, out[4] = p.whole, out[5] = p.rotates;
}

// The segments of workgroup x0 of n along the list, five ints each (sequence, first tile, end tile,
// part, parts); at most `room` of them.  Returns their number, -1 where the lanes disagree, -2
// beyond `room`.
int host_segments(const int32_t *seq_lens, int batch, int num_splits, int sw, int per_seq, int n, int x0, int *out,
                  int room) {
    args.seq_lens = seq_lens;
    args.batch = batch;
    args.num_splits = num_splits;
    args.sw = sw;
    args.per_seq = per_seq;
    nx = n;
    x = x0;
    lanes::run(one_lane);
    tq4::xdl::Cut c = cuts[0];
    for (int l = 1; l < lanes::kLanes; ++l)
        if (found[l] != found[0] || single[l] != single[0] ||
            (found[0] && (cuts[l].b != c.b || cuts[l].len != c.len || cuts[l].run.first != c.run.first ||
                          cuts[l].run.count != c.run.count || cuts[l].p != c.p || cuts[l].n_parts != c.n_parts)))
            return -1;
    int k = 0;
    for (bool more = found[0]; more; more = !single[0] && tq4::xdl::next_segment(c, args, x, true)) {
        if (k == room)
            return -2;
        int *o = out + 5 * k++;
        o[0] = c.b, o[1] = c.run.first, o[2] = c.run.first + c.run.count, o[3] = c.p, o[4] = c.n_parts;
    }
    return k;
}

// Run i of n over `tiles` tiles.
void host_run(int tiles, int n, int i, int *first, int *count) {
    const auto r = tq4::xdl::run_of(tiles, n, i);
    *first = r.first;
    *count = r.count;
}

int host_waves(void) { return tq4::xdl::kStepWaves; }
}
