// Batched CG / Jacobi-PCG of systems with short, banded rows, each solved by a
// team of workgroups that keeps it on the CUs from the first iteration to the
// last.
//
// The per-kernel batch runs three kernels per iteration over all systems until
// the slowest has converged: on 48 systems of 1,000 to 60,000 rows 730 iterations
// of 20 us, launch latency and one wavefront per system deciding.  Here a system
// of n rows gets ceil(n / piece) workgroups of 1,024 lanes with R rows each:
// vectors and row entries in registers, u of the piece and of the `halo` rows on
// either side in LDS.  A team exchanges u's rows near its pieces' ends and four
// sums per iteration as tagged 64-bit words (persist.hip), every workgroup of it
// decides alike, and teams never wait for each other, so a stopped system frees
// its CUs' bandwidth at once.  Teams that do not fit the chip together run in
// successive cooperative launches, largest systems first, so that a launch's systems
// are of like length; the one-workgroup systems past the last of them wait for nobody
// and run in one ordinary launch (in cooperative ones of 256, each 130 us before its
// first iteration, 2,048 systems of 1,000 FP32 rows took 2.93 ms for 100 iterations;
// now 2.11, in the kernels 7.5).
//
// The iteration is that of the per-kernel batch (BatchState::advance); its dot
// products are summed per workgroup and then per team instead of per 64-row
// chunk.
#include "persist_batch.hpp"

#include <algorithm>
#include <numeric>
#include <type_traits>

#include "persist_launch.hpp"
#include "tuning.hpp"

namespace pm
{
namespace
{

constexpr int kTeamEntries = 8;    // row entries in registers
constexpr int kTeamSlots = 256;    // workgroups of a launch at most
constexpr int kTeamLargest = kWave; // workgroups of a team: one lane each in the decision
constexpr int32_t kTeamIterations = 1 << 16;  // a launch runs a system to its end

// One workgroup's part of a launch.
struct TeamTask
{
    int32_t system, slot0, team, piece;  // its team's first workgroup and size, its piece
    int32_t rows, halo;                  // of the system
    int64_t begin;                       // the system's first row
};

struct TeamControl
{
    unsigned abort;
    unsigned pad[63];
    unsigned finished[kTeamSlots];       // workgroups of a team (by first slot) that reached the end
    BatchState out[kTeamSlots];          // ... and its final state
    TeamTask tasks[kTeamSlots];
    word part[2][kCgValues][2][kTeamSlots];
};

template <typename S, typename I>
struct TeamArgs
{
    const I* ro;
    const I* ci;
    const S* values;
    const S* rhs;
    const S* x;
    S* x_out;
    const S *p, *r, *s, *w;
    const S* inv;
    const BatchState* st;
    const TeamTask* tasks;
    TeamControl* ctl;
    word* xu;                 // [slot][row of the piece]
    word* xx;
    int plane;                // words of a half plane
    unsigned tag;
    int32_t max_iterations;
    int refresh;
    BatchState* end;                 // teams of one workgroup: the states and the count of stopped
    unsigned long long* done_count;  // systems, which they write themselves (null: k_team_states)
};

template <typename S, typename I, int R>
__global__ __launch_bounds__(kPersistThreads) void k_batch_team(TeamArgs<S, I> a)
{
    using X = Exchange<S>;
    constexpr int E = kTeamEntries;
    constexpr int kPiece = R * kPersistThreads;
    extern __shared__ char lds_raw[];
    __shared__ double lds_p[kCgValues][kPersistWaves];
    __shared__ BatchState state;
    __shared__ S sh_alpha, sh_beta;
    __shared__ int sh_code, sh_fail;

    const int tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
    const TeamTask job = a.tasks[blockIdx.x];
    const int H = job.team > 1 ? job.halo : 0;
    const int first = job.piece * kPiece;  // the piece's first row of the system
    const int size = job.rows - first < kPiece ? job.rows - first : kPiece;
    const int words0 = job.slot0 * kPiece;  // the system's rows in the exchange
    S* us = reinterpret_cast<S*>(lds_raw);  // u of rows [first - H, first + kPiece + H)

    S p[R], s[R], x[R], r[R], w[R], inv[R], val[R][E];
    unsigned col[R][E / 2];  // two 16-bit places in us each
#pragma unroll
    for (int k = 0; k < R; ++k)
    {
        const int l = k * kPersistThreads + tid;
        const bool ok = l < size;
        const int64_t i = job.begin + first + (ok ? l : 0);
        p[k] = ok ? a.p[i] : S(0);
        s[k] = ok ? a.s[i] : S(0);
        x[k] = ok ? a.x[i] : S(0);
        r[k] = ok ? a.r[i] : S(0);
        w[k] = ok ? a.w[i] : S(0);
        inv[k] = !ok ? S(0) : a.inv != nullptr ? a.inv[i] : S(1);
        const int64_t b = static_cast<int64_t>(a.ro[i]);
        const int n = ok ? static_cast<int>(static_cast<int64_t>(a.ro[i + 1]) - b) : 0;
#pragma unroll
        for (int e = 0; e < E; ++e)
        {
            // an absent entry is 0 times the row's own u
            val[k][e] = e < n ? a.values[b + e] : S(0);
            const int c = e < n ? static_cast<int>(static_cast<int64_t>(a.ci[b + e]) - job.begin) - first : (ok ? l : 0);
            const unsigned at = static_cast<unsigned>(c + H);
            if (e % 2 == 0) col[k][e / 2] = at;
            else col[k][e / 2] |= at << 16;
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    // halo rows past the system stay 0
    for (int q = tid; q < kPiece + 2 * H; q += kPersistThreads) us[q] = S(0);
    if (tid == 0)
    {
        state = a.st[job.system];
        sh_alpha = static_cast<S>(state.alpha);
        sh_beta = static_cast<S>(state.beta);
        sh_code = state.done;
        sh_fail = given_up(&a.ctl->abort);
    }
    __syncthreads();
    if (sh_fail != 0) return;
    auto u_of = [&](int k) { return inv[k] * r[k]; };

    auto publish = [&](word* buf, unsigned tag, auto get) {
#pragma unroll
        for (int k = 0; k < R; ++k)
        {
            const int l = k * kPersistThreads + tid;
            if (l >= size) continue;
            const S v = get(k);
            us[H + l] = v;
            if (l < H || l >= size - H) X::put(buf, a.plane, words0 + first + l, v, tag);
        }
    };
    // acc[k] = row k of A v for the vector published last, entries left to right
    auto product = [&](const word* buf, unsigned tag, auto* acc) {
        using Acc = std::remove_reference_t<decltype(acc[0])>;
        bool fine = true;
        for (int h0 = 0; h0 < 2 * H; h0 += kPersistThreads)
        {
            const int h = h0 + tid;
            const int q = h < H ? h - H : size + (h - H);
            const int i = first + q;
            if (h >= 2 * H || i < 0 || i >= job.rows) continue;
            word hw[X::kWords];
            fine = wait_for(&a.ctl->abort, [&] {
                       X::issue(buf, a.plane, words0 + i, hw);
                       return ready<S>(hw, tag);
                   }) && fine;
            us[H + q] = X::value(hw);
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < R; ++k)
        {
            Acc sum = Acc(0);
#pragma unroll
            for (int e = 0; e < E; ++e)
            {
                const unsigned at = e % 2 == 0 ? col[k][e / 2] & 0xffffu : col[k][e / 2] >> 16;
                sum = fma_s<Acc>(static_cast<Acc>(val[k][e]), static_cast<Acc>(us[at]), sum);
            }
            acc[k] = k * kPersistThreads + tid < size ? sum : Acc(0);
            if (R > 2) __builtin_amdgcn_sched_barrier(0);
        }
        if (!fine) sh_fail = 1;
    };

    unsigned tag = a.tag;
    for (int t = 0; sh_code == kRunning; ++t)
    {
        ++tag;
        const S al = sh_alpha, be = sh_beta;
        const bool refresh = a.refresh > 0 && (t + 1) % a.refresh == 0;
#pragma unroll
        for (int k = 0; k < R; ++k)
        {
            p[k] = fma_s(be, p[k], u_of(k));
            s[k] = fma_s(be, s[k], w[k]);
            x[k] = fma_s(al, p[k], x[k]);
            if (!refresh) r[k] = fma_s(-al, s[k], r[k]);
        }
        if (refresh)
        {
            // r = b - A x with FP64 accumulation
            publish(a.xx, tag, [&](int k) { return x[k]; });
            double ax[R];
            product(a.xx, tag, ax);
#pragma unroll
            for (int k = 0; k < R; ++k)
            {
                const int l = k * kPersistThreads + tid;
                if (l < size) r[k] = static_cast<S>(static_cast<double>(a.rhs[job.begin + first + l]) - ax[k]);
            }
            __syncthreads();
        }
        publish(a.xu, tag, u_of);
        product(a.xu, tag, w);

        double part[kCgValues] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int k = 0; k < R; ++k)
        {
            const double rv = static_cast<double>(r[k]), uv = static_cast<double>(u_of(k));
            part[0] = __builtin_fma(rv, rv, part[0]);
            part[1] = __builtin_fma(rv, uv, part[1]);
            part[2] = __builtin_fma(static_cast<double>(w[k]), uv, part[2]);
            part[3] = __builtin_fma(uv, static_cast<double>(s[k]), part[3]);
        }
        const double wsum = wave_sum4(part[0], part[1], part[2], part[3]);
        if (lane % 16 == 0) lds_p[lane / 16][wave] = wsum;
        __syncthreads();
        if (sh_fail != 0) return;
        if (wave == 0)
        {
            // row v of the wavefront sums value v over the wavefronts
            double mine = lds_p[lane / 16][lane % 16];
            mine = butterfly_add<8>(mine);
            mine = butterfly_add<4>(mine);
            mine = butterfly_add<2>(mine);
            mine = butterfly_add<1>(mine);
            double tot[kCgValues];
            bool fine = true;
            if (job.team > 1)
            {
                if (lane % 16 == 0)
                    Exchange<double>::put(&a.ctl->part[t & 1][lane / 16][0][blockIdx.x], kTeamSlots, 0, mine, tag);
                double v[kCgValues] = {0.0, 0.0, 0.0, 0.0};
                if (lane < job.team)
                {
                    const word* from = &a.ctl->part[t & 1][0][0][job.slot0 + lane];
                    word hw[kCgValues][2];
                    fine = wait_for(&a.ctl->abort, [&] {
                        bool ok = true;
#pragma unroll
                        for (int q = 0; q < kCgValues; ++q)
                        {
                            hw[q][0] = load_word(from + (2 * q) * kTeamSlots);
                            hw[q][1] = load_word(from + (2 * q + 1) * kTeamSlots);
                        }
#pragma unroll
                        for (int q = 0; q < kCgValues; ++q)
                            ok = ok && word_ready(hw[q][0], tag) && word_ready(hw[q][1], tag);
                        return ok;
                    });
#pragma unroll
                    for (int q = 0; q < kCgValues; ++q) v[q] = Exchange<double>::value(hw[q]);
                }
                mine = wave_sum4(v[0], v[1], v[2], v[3]);
            }
#pragma unroll
            for (int q = 0; q < kCgValues; ++q) tot[q] = __shfl(mine, q * 16, kWave);
            if (!fine) sh_fail = 1;
            if (lane == 0)
            {
                sh_code = state.template advance<S>(tot[0], tot[1], tot[2], tot[3], a.max_iterations);
                sh_alpha = static_cast<S>(state.alpha);
                sh_beta = static_cast<S>(state.beta);
            }
        }
        __syncthreads();
        if (sh_fail != 0) return;
    }

#pragma unroll
    for (int k = 0; k < R; ++k)
    {
        const int l = k * kPersistThreads + tid;
        if (l < size) a.x_out[job.begin + first + l] = x[k];
    }
    BatchState end = state;
    end.done = sh_code;
    if (a.end != nullptr)
    {
        // no workgroup but this one can fail the system
        if (tid != 0 || a.st[job.system].done != kRunning) return;  // stopped before the launch, and counted then
        a.end[job.system] = end;
        atomicAdd(a.done_count, 1ull);
        return;
    }
    if (tid == 0 && job.piece == 0) a.ctl->out[job.slot0] = end;
    __syncthreads();
    if (tid == 0)
        __hip_atomic_fetch_add(&a.ctl->finished[job.slot0], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The x of every team whose workgroups all reached the end, then (in a kernel of
// its own) its state.
template <typename S>
__global__ __launch_bounds__(kBlock) void k_team_commit(const TeamControl* ctl, int piece_rows,
                                                        const S* __restrict__ from, S* __restrict__ x)
{
    const TeamTask job = ctl->tasks[blockIdx.x];
    if (ctl->finished[job.slot0] != static_cast<unsigned>(job.team)) return;
    const int first = job.piece * piece_rows;
    const int size = job.rows - first < piece_rows ? job.rows - first : piece_rows;
    for (int l = threadIdx.x; l < size; l += kBlock) x[job.begin + first + l] = from[job.begin + first + l];
}

// *gave_up = 1 (host memory) when the launch was left unfinished.
__global__ void k_team_states(const TeamControl* ctl, int slots, BatchState* st, unsigned long long* done_count,
                              unsigned* gave_up)
{
    const int slot = static_cast<int>(threadIdx.x);
    if (slot == 0 && ctl->abort != 0u) *gave_up = 1u;
    if (slot >= slots) return;
    const TeamTask job = ctl->tasks[slot];
    if (job.piece != 0 || ctl->finished[slot] != static_cast<unsigned>(job.team)) return;
    if (st[job.system].done != kRunning) return;  // stopped before the launch, and counted then
    st[job.system] = ctl->out[slot];
    atomicAdd(done_count, 1ull);
}

// `before`: the call's launch before this one (or null); after one that gave up the
// next ones do too, so that a call waits for one of them at most.
__global__ void k_team_reset(TeamControl* ctl, const TeamControl* before, unsigned abort)
{
    if (threadIdx.x == 0) ctl->abort = before != nullptr && before->abort != 0u ? 1u : abort;
    if (threadIdx.x < kTeamSlots) ctl->finished[threadIdx.x] = 0u;
}

// The band of every system of short rows, kNoBand for the others: rows too long, a
// column outside the system, or more than `largest` rows.  A wavefront takes
// consecutive 64-row chunks and tells a system's value once per run of its chunks
// (once per chunk, 24,752 chunks of 8 systems met on one cache line: five iterations of
// eight 198,000-row FP32 systems 1.02 ms, now 0.49).
constexpr int kNoBand = 0x7fffffff;
constexpr int kLookWaves = 2048;
template <typename I>
__global__ __launch_bounds__(kBlock) void k_team_look(int64_t chunks, const int32_t* __restrict__ chunk_sys,
                                                      const int64_t* __restrict__ sys_end,
                                                      const int64_t* __restrict__ sys_chunk0,
                                                      const I* __restrict__ ro, const I* __restrict__ ci,
                                                      int64_t largest, BatchLook* look)
{
    const int64_t waves = static_cast<int64_t>(gridDim.x) * (kBlock / kWave);
    const int64_t per = (chunks + waves - 1) / waves;
    const int64_t wave = static_cast<int64_t>(blockIdx.x) * (kBlock / kWave) + threadIdx.x / kWave;
    const int64_t c1 = (wave + 1) * per < chunks ? (wave + 1) * per : chunks;
    int32_t now = -1;
    int band = 0;
    auto tell = [&]() {
        if (now < 0) return;
#pragma unroll
        for (int off = kWave / 2; off > 0; off /= 2) band = max(band, __shfl_xor(band, off, kWave));
        if (threadIdx.x % kWave == 0) atomicMax(&look[now].band, band);
    };
    for (int64_t c = wave * per; c < c1; ++c)
    {
        const int32_t s = chunk_sys[c];
        if (s != now)
        {
            tell();
            now = s;
            band = 0;
        }
        if (s < 0) continue;
        const int64_t row = c * kChunkRows + threadIdx.x % kWave;
        const int64_t begin = sys_chunk0[s] * kChunkRows, end = sys_end[s];
        if (end - begin > largest) band = kNoBand;
        if (row >= end || band == kNoBand) continue;
        const int64_t b = static_cast<int64_t>(ro[row]), e = static_cast<int64_t>(ro[row + 1]);
        if (e - b > kTeamEntries) band = kNoBand;
        else
            for (int64_t k = b; k < e; ++k)
            {
                const int64_t col = static_cast<int64_t>(ci[k]);
                // a system has at most 2^18 rows here
                if (col < begin || col >= end) band = kNoBand;
                else band = max(band, static_cast<int>(col < row ? row - col : col - row));
            }
    }
    tell();
}

__global__ void k_look_reset(int64_t systems, BatchLook* look)
{
    for (int64_t s = threadIdx.x; s < systems; s += blockDim.x) look[s] = BatchLook{0};
}

size_t team_lds(int es, int rows_per_lane, int halo)
{
    return static_cast<size_t>(es) * (static_cast<size_t>(rows_per_lane) * kPersistThreads + 2 * static_cast<size_t>(halo));
}

template <typename S, typename I>
const void* team_kernel(int rows_per_lane)
{
    if (rows_per_lane == 1) return reinterpret_cast<const void*>(k_batch_team<S, I, 1>);
    if (rows_per_lane == 2) return reinterpret_cast<const void*>(k_batch_team<S, I, 2>);
    if constexpr (sizeof(S) == 4) return reinterpret_cast<const void*>(k_batch_team<S, I, 4>);
    return nullptr;
}

// Systems below kTinyBytes of a vector leave most lanes of a workgroup idle: more than
// kTinyRounds of them for every CU take the kernels.  60 iterations of FP32 systems,
// kernels / a workgroup each: 1,024 of 64 rows 1.17 / 0.87 ms, 2,048 of 128 rows 1.67 /
// 2.20, 8,192 of 64 rows 4.6 / 8.4, 2,048 of 256 rows 2.16 / 1.56; FP64, 8,192 of 64
// rows 4.7 / 7.2, of 128 rows 6.24 / 6.09.
constexpr int64_t kTinyBytes = 1024;
constexpr int64_t kTinyRounds = 4;

// Rows of a system that teams take, at least.
int64_t least_rows(const BatchTeams& b, int es, int slots)
{
    int64_t tiny = 0;
    for (int64_t s = 0; s < b.systems; ++s) tiny += (b.end[s] - b.begin[s]) * es < kTinyBytes;
    return tiny > kTinyRounds * slots ? kTinyBytes / es : 1;
}

// The tasks of one-workgroup systems, behind the looks.
size_t team_tasks_offset(int64_t systems)
{
    return (sizeof(BatchLook) * static_cast<size_t>(systems) + 255) & ~size_t(255);
}

// Rows per lane that the registers hold.
template <typename S>
constexpr int team_rows()
{
    return sizeof(S) == 4 ? 4 : 2;
}

// Workgroups of a launch at most; 0: no teams.
int team_slots(const pm_workspace* ws, const BatchTeams& b, int* slots)
{
    *slots = 0;
    if (!persist_enabled() || !persist_resident(ws, 1) || b.max_iterations > kTeamIterations) return PM_OK;
    int cus = 0;
    PM_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, ws->device));
    *slots = std::min(cus, kTeamSlots);
    return PM_OK;
}

template <typename S, typename I>
int teams_run(pm_workspace* ws, const BatchTeams& b, const std::vector<BatchLook>& look, const I* ro, const I* ci,
              hipStream_t stream, bool* ran)
{
    *ran = false;
    const int most = team_rows<S>();
    const int es = static_cast<int>(sizeof(S));
    int slots = 0;
    PM_TRY(team_slots(ws, b, &slots));
    const int64_t least = least_rows(b, es, slots);
    std::vector<int> order;
    int64_t total[3] = {0, 0, 0};  // workgroups with 1, 2, 4 rows per lane
    for (int64_t s = 0; s < b.systems; ++s)
    {
        const int64_t n = b.end[s] - b.begin[s];
        const BatchLook& l = look[static_cast<size_t>(s)];
        const int64_t piece = static_cast<int64_t>(most) * kPersistThreads;
        const int64_t team = ceil_div(n, piece);
        if (n < least || b.skip[s] || l.band == kNoBand || team > std::min(kTeamLargest, slots)) continue;
        if (team > 1 && (team_lds(es, most, l.band) > kPersistLds || piece + 2 * static_cast<int64_t>(l.band) > 65535)) continue;
        order.push_back(static_cast<int>(s));
        for (int k = 0; k < 3; ++k) total[k] += ceil_div(n, static_cast<int64_t>(kPersistThreads) << k);
    }
    if (order.empty()) return PM_OK;
    *ran = true;
    // as few rows per lane as let all teams run together (and no team grow past
    // its decision's lanes)
    int rows_per_lane = most;
    for (int k = 0; (1 << k) < most; ++k)
    {
        bool fits = total[k] <= slots;
        for (int s : order)
        {
            const int64_t piece = static_cast<int64_t>(kPersistThreads) << k;
            fits = fits && ceil_div(b.end[s] - b.begin[s], piece) <= kTeamLargest;
        }
        if (fits)
        {
            rows_per_lane = 1 << k;
            break;
        }
    }
    const int64_t piece = static_cast<int64_t>(rows_per_lane) * kPersistThreads;
    std::stable_sort(order.begin(), order.end(),
                     [&](int l, int r) { return b.end[l] - b.begin[l] > b.end[r] - b.begin[r]; });
    // launches of at most `slots` workgroups, which run together
    std::vector<std::vector<TeamTask>> launches;
    std::vector<TeamTask> now;
    const bool together = total[rows_per_lane / 2] <= slots;
    auto add = [&](int s) {
        const int64_t n = b.end[s] - b.begin[s];
        const int team = static_cast<int>(ceil_div(n, piece));
        if (static_cast<int>(now.size()) + team > slots) return false;
        const int slot0 = static_cast<int>(now.size());
        for (int q = 0; q < team; ++q)
            now.push_back(TeamTask{s, slot0, team, q, static_cast<int32_t>(n), look[static_cast<size_t>(s)].band, b.begin[s]});
        return true;
    };
    // ... up to the last one with a system of several workgroups; the smaller systems
    // that it has no room for wait for nobody
    size_t at = 0;
    for (; at < order.size(); ++at)
    {
        const int64_t n = b.end[order[at]] - b.begin[order[at]];
        if ((together || n > piece || !now.empty()) && add(order[at])) continue;
        if (!now.empty()) launches.push_back(std::move(now));
        now.clear();
        if (n <= piece) break;
        (void)add(order[at]);
    }
    if (!now.empty()) launches.push_back(std::move(now));
    std::vector<TeamTask> alone[3];  // by 1, 2, 4 rows per lane
    for (; at < order.size(); ++at)
    {
        const int s = order[at];
        const int64_t n = b.end[s] - b.begin[s];
        const int k = n <= kPersistThreads ? 0 : n <= 2 * kPersistThreads ? 1 : 2;
        alone[k].push_back(TeamTask{s, 0, 1, 0, static_cast<int32_t>(n), 0, b.begin[s]});
    }

    const size_t words = static_cast<size_t>(slots) * static_cast<size_t>(piece);
    const size_t plane_words = words * Exchange<S>::kWords;
    const size_t control = (sizeof(TeamControl) + 255) & ~size_t(255);
    const size_t control_all = control * std::max<size_t>(launches.size(), 1);
    // the control blocks come after the words, whose places then only ever hold words
    const size_t need = 2 * plane_words * sizeof(word) + control_all;
    // (blocks in a place that earlier held words, or the other way round, are
    // cleared with the whole buffer when the layout changes)
    ws->teams_tag = static_cast<uint32_t>(persist_test("tag=", ws->teams_tag));
    const uint64_t tags = launches.size() * (static_cast<uint64_t>(b.max_iterations) + 2u);
    if (tags > kLastTag) return PM_OK;
    if (need > ws->teams.bytes || ws->teams_words != plane_words || ws->teams_tag + tags > kLastTag)
    {
        if (!persist_storage(ws->teams, need))
        {
            ws->last_one_launch = -1;
            return PM_OK;
        }
        hipLaunchKernelGGL(k_persist_clear, dim3(1024), dim3(kBlock), 0, stream, ws->teams.as<word>(),
                           static_cast<int64_t>(ws->teams.bytes / sizeof(word)));
        PM_HIP(hipGetLastError());
        ws->teams_words = plane_words;
        ws->teams_tag = 0;
    }
    const void* kernel = team_kernel<S, I>(rows_per_lane);
    TeamArgs<S, I> a{};
    a.ro = ro;
    a.ci = ci;
    a.values = static_cast<const S*>(b.a->values);
    a.rhs = static_cast<const S*>(b.rhs);
    a.x = static_cast<const S*>(b.x);
    a.x_out = static_cast<S*>(b.x_out);
    a.p = static_cast<const S*>(b.p);
    a.r = static_cast<const S*>(b.r);
    a.s = static_cast<const S*>(b.s);
    a.w = static_cast<const S*>(b.w);
    a.inv = static_cast<const S*>(b.inv);
    a.st = b.st;
    a.xu = ws->teams.as<word>();
    a.xx = a.xu + plane_words;
    a.plane = static_cast<int>(words);
    a.max_iterations = b.max_iterations;
    a.refresh = b.refresh;
    // the tasks of every launch in one synchronous copy (the host arrays go out of scope)
    char* blocks0 = ws->teams.as<char>() + 2 * plane_words * sizeof(word);
    for (size_t k = 0; k < launches.size(); ++k)
    {
        auto* ctl = reinterpret_cast<TeamControl*>(blocks0 + k * control);
        PM_HIP(hipMemcpyAsync(ctl->tasks, launches[k].data(), sizeof(TeamTask) * launches[k].size(),
                              hipMemcpyHostToDevice, stream));
    }
    unsigned* gave_up = &ws->host_state[0].counters[0];
    *gave_up = 0u;
    ws->last_one_launch = 1;
    const TeamControl* before = nullptr;
    for (size_t k = 0; k < launches.size(); ++k)
    {
        auto* ctl = reinterpret_cast<TeamControl*>(blocks0 + k * control);
        const int grid = static_cast<int>(launches[k].size());
        int halo = 0;
        for (const TeamTask& t : launches[k]) halo = std::max(halo, t.team > 1 ? t.halo : 0);
        const size_t lds = team_lds(es, rows_per_lane, halo);
        PM_TRY(persist_allow_lds(kernel));
        a.tasks = ctl->tasks;
        a.ctl = ctl;
        a.tag = ws->teams_tag;
        ws->teams_tag += static_cast<uint32_t>(b.max_iterations) + 2u;
        hipLaunchKernelGGL(k_team_reset, dim3(1), dim3(kTeamSlots), 0, stream, ctl, before,
                           persist_test("give_up=", -1) == static_cast<int64_t>(k) ? 1u : 0u);
        before = ctl;
        PM_HIP(hipGetLastError());
        void* args[] = {&a};
        const hipError_t err = persist_launch(kernel, grid, args, lds, stream, static_cast<int64_t>(k));
        if (persist_refused(err, ws))
        {
            ws->last_one_launch = -1;
            break;
        }
        PM_HIP(err);
        hipLaunchKernelGGL(k_team_commit<S>, dim3(grid), dim3(kBlock), 0, stream, ctl, static_cast<int>(piece),
                           static_cast<const S*>(b.x_out), static_cast<S*>(b.x));
        hipLaunchKernelGGL(k_team_states, dim3(1), dim3(kTeamSlots), 0, stream, ctl, grid, b.st, b.done_count,
                           gave_up);
        PM_HIP(hipGetLastError());
    }
    a.ctl = reinterpret_cast<TeamControl*>(blocks0);
    a.x_out = static_cast<S*>(b.x);
    a.end = b.st;
    a.done_count = b.done_count;
    auto* tasks = reinterpret_cast<TeamTask*>(ws->looks.as<char>() + team_tasks_offset(b.systems));
    for (int k = 0; k < 3; ++k)
    {
        if (alone[k].empty()) continue;
        PM_HIP(hipMemcpyAsync(tasks, alone[k].data(), sizeof(TeamTask) * alone[k].size(), hipMemcpyHostToDevice, stream));
        hipLaunchKernelGGL(k_team_reset, dim3(1), dim3(kTeamSlots), 0, stream, a.ctl, nullptr, 0u);
        a.tasks = tasks;
        tasks += alone[k].size();
        const void* one = team_kernel<S, I>(1 << k);
        const size_t lds = team_lds(es, 1 << k, 0);
        PM_TRY(persist_allow_lds(one));
        void* args[] = {&a};
        PM_HIP(hipLaunchKernel(one, dim3(static_cast<unsigned>(alone[k].size())), dim3(kPersistThreads), args, lds, stream));
    }
    // the vectors of tasks are the sources of the copies above
    PM_HIP(hipStreamSynchronize(stream));
    if (*gave_up != 0u)
    {
        ws->persist_pause = kPersistPause;
        ws->last_one_launch = -1;
    }
    return PM_OK;
}

} // namespace

int batch_teams_look(pm_workspace* ws, const BatchTeams& b, std::vector<BatchLook>& look, hipStream_t stream)
{
    look.assign(static_cast<size_t>(b.systems), BatchLook{kNoBand});  // none fits
    int slots = 0;
    PM_TRY(team_slots(ws, b, &slots));
    const int64_t piece = static_cast<int64_t>(b.a->dtype == PM_F64 ? team_rows<double>() : team_rows<float>()) * kPersistThreads;
    const int64_t largest = piece * std::min(kTeamLargest, slots);
    const int64_t least = least_rows(b, b.a->dtype == PM_F64 ? 8 : 4, slots);
    bool any = false;
    for (int64_t s = 0; s < b.systems && !any; ++s)
        any = !b.skip[s] && b.end[s] - b.begin[s] >= least && b.end[s] - b.begin[s] <= largest;
    if (!any || b.chunks == 0) return PM_OK;
    if (!persist_storage(ws->looks, team_tasks_offset(b.systems) + sizeof(TeamTask) * static_cast<size_t>(b.systems)))
    {
        ws->last_one_launch = -1;
        return PM_OK;
    }
    auto* dev = ws->looks.as<BatchLook>();
    hipLaunchKernelGGL(k_look_reset, dim3(1), dim3(kBlock), 0, stream, b.systems, dev);
    const dim3 grid(static_cast<unsigned>(ceil_div(std::min<int64_t>(b.chunks, kLookWaves), kBlock / kWave)));
    if (use_compact(b.a))
        hipLaunchKernelGGL(k_team_look<int32_t>, grid, dim3(kBlock), 0, stream, b.chunks, b.chunk_sys, b.sys_end,
                           b.sys_chunk0, b.a->row_offsets32, b.a->col_indices32, largest, dev);
    else
        hipLaunchKernelGGL(k_team_look<int64_t>, grid, dim3(kBlock), 0, stream, b.chunks, b.chunk_sys, b.sys_end,
                           b.sys_chunk0, b.a->row_offsets, b.a->col_indices, largest, dev);
    PM_HIP(hipGetLastError());
    PM_HIP(hipMemcpyAsync(look.data(), dev, sizeof(BatchLook) * look.size(), hipMemcpyDeviceToHost, stream));
    PM_HIP(hipStreamSynchronize(stream));
    return PM_OK;
}

int batch_teams_run(pm_workspace* ws, const BatchTeams& b, const std::vector<BatchLook>& look, hipStream_t stream,
                    bool* ran)
{
    const pm_csr* m = b.a;
    const bool compact = use_compact(m);
    if (m->dtype == PM_F64)
        return compact ? teams_run<double>(ws, b, look, m->row_offsets32, m->col_indices32, stream, ran)
                       : teams_run<double>(ws, b, look, m->row_offsets, m->col_indices, stream, ran);
    return compact ? teams_run<float>(ws, b, look, m->row_offsets32, m->col_indices32, stream, ran)
                   : teams_run<float>(ws, b, look, m->row_offsets, m->col_indices, stream, ran);
}

} // namespace pm
