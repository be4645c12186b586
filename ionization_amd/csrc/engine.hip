// Native runtime of the mesh-TDSE library: context, device memory pool,
// ragged work tables, hipGraph-captured steps and the C ABI of tdse_hip.h.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <array>
#include <cmath>
#include <cstddef>
#include <cstdio>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/tdse_hip.h"
#include "common.h"
#include "cyl_kernels.h"
#include "line_kernels.h"
#include "sh_kernels.h"
#include "tdma_kernels.h"

namespace {

constexpr int kAbiVersion = 1;
constexpr size_t kAlign = 256;
// Steps captured in the longer of the two step graphs (runs of at least this
// many steps replay it; the rest replay the one-step graph): one launch per 8
// steps took small batches 6-9 % faster (one 200 x 1000 SH simulation: 0.047 ->
// 0.043 ms/step) and changed nothing for the 256-simulation scan.
constexpr int kGraphSteps = 8;
constexpr int kMaxL = 4096;          // largest l_bound accepted (c_l table size)
constexpr int kSlotCapacity = 8192;  // simulations of each kind per context
constexpr int kSideStreams = 3;      // extra streams for concurrent R-phase buckets (default priority)
constexpr int kMaxRidingJobs = 1024;  // observation jobs (one wave each) that ride in an R-phase launch
constexpr int kMaxPairThreads = 512; // largest workgroup of the two-line (velocity odd l-pair) R-phase
constexpr int kNoObs = -1;           // no observation partials of a freshly uploaded cylindrical state
constexpr int kNoFlags = 0;          // health flags of a freshly uploaded state
static_assert(TDSE_FLAG_NONFINITE == TDSE_HEALTH_NONFINITE && TDSE_FLAG_NORM_GROWTH == TDSE_HEALTH_NORM_GROWTH,
              "health flag values of the ABI and the kernels differ");

thread_local std::string g_lib_error;

// First-fit sub-allocator over one device buffer reserved at context creation.
class Arena {
   public:
    char* base = nullptr;
    size_t size = 0;
    size_t used = 0;

    // beyond: a block of `extra` bytes past the pool, from the same allocation (null where only the pool itself fits)
    char* beyond = nullptr;
    bool init(size_t bytes, size_t extra) {
        size = (bytes + kAlign - 1) / kAlign * kAlign;
        if (hipMalloc(&base, size + extra) == hipSuccess) {
            beyond = base + size;
        } else {
            (void)hipGetLastError();  // not the next launch's
            if (hipMalloc(&base, size) != hipSuccess) {
                base = nullptr;
                return false;
            }
        }
        free_[0] = size;
        return true;
    }
    void release() {
        if (base) (void)hipFree(base);
        base = beyond = nullptr;
    }
    // Returns nullptr when no free block is large enough.
    void* alloc(size_t bytes) {
        bytes = std::max<size_t>(kAlign, (bytes + kAlign - 1) / kAlign * kAlign);
        for (auto it = free_.begin(); it != free_.end(); ++it) {
            if (it->second >= bytes) {
                const size_t off = it->first;
                const size_t rest = it->second - bytes;
                free_.erase(it);
                if (rest) free_[off + bytes] = rest;
                used_[off] = bytes;
                used += bytes;
                return base + off;
            }
        }
        return nullptr;
    }
    void dealloc(void* p) {
        if (!p) return;
        const size_t off = static_cast<char*>(p) - base;
        auto it = used_.find(off);
        if (it == used_.end()) return;
        size_t sz = it->second;
        used -= sz;
        used_.erase(it);
        size_t start = off;
        auto next = free_.lower_bound(off);
        if (next != free_.end() && next->first == off + sz) {
            sz += next->second;
            free_.erase(next);
        }
        auto prev = free_.lower_bound(off);
        if (prev != free_.begin()) {
            --prev;
            if (prev->first + prev->second == off) {
                start = prev->first;
                sz += prev->second;
                free_.erase(prev);
            }
        }
        free_[start] = sz;
    }

   private:
    std::map<size_t, size_t> free_;
    std::map<size_t, size_t> used_;
};

struct ShHost {
    bool live = false;
    bool vel = false;    // velocity gauge (one more table row, h2 factors around the R-phase)
    bool adi = false;    // AlternatingDirectionImplicit (its own r and l sweeps instead of the R-phase)
    ShSim dev{};
    int n_data = 0;
    int wave_first = 0;  // this simulation's range in the wave table
    int wave_count = 0;
    std::vector<void*> blocks;
};

struct LineHost {
    bool live = false;
    bool complex_steps = false;  // some w_n has a nonzero real part
    LineSim dev{};
    int n_data = 0;
    std::vector<void*> blocks;
};

struct CylHost {
    bool live = false;
    CylSim dev{};
    int n_data = 0;
    std::vector<void*> blocks;
};

// Device table with host-side growth.
template <class T>
struct DevVec {
    T* ptr = nullptr;
    size_t cap = 0;
    size_t count = 0;
};

struct Bucket {
    int M = 0;  // exact rows per chunk-thread
    int P = 0;
    bool imag = false;  // Line: complex time steps (imaginary-time relaxation)
    int method = 0;     // Line: LINE_ADI, LINE_SIO_LEN or LINE_SIO_VEL
    size_t lds = 0;     // Line, M == 0 (any layouts): dynamic LDS of the launch
    int Mr = 0, Cr = 0, lanes = 1;  // cylindrical rho-sweep: rows per thread, chunks, lines per workgroup
    DevVec<int2> lines;   // SH: (slot, l); Line: (slot, 0); Cyl z-sweep: (slot, pair of rho-lines)
    DevVec<int2> rlines;  // Cyl rho-sweep: (slot, position group)
    DevVec<int2> vpairs[2];  // SH: the velocity-gauge l-pairs (slot, l) of even / odd l among these simulations
    DevVec<int2> fpairs;     // SH: velocity-gauge odd l-pairs solved with their h2 factors (k_sh_rphase_vpair)
};

void free_bucket(Bucket& b) {
    if (b.lines.ptr) (void)hipFree(b.lines.ptr);
    if (b.rlines.ptr) (void)hipFree(b.rlines.ptr);
    for (auto& v : b.vpairs)
        if (v.ptr) (void)hipFree(v.ptr);
    if (b.fpairs.ptr) (void)hipFree(b.fpairs.ptr);
    b = Bucket{};
}

// Norm partials along l of one simulation (kShPartRows rows each).
int sh_parts(int L) { return (L + kShPartRows - 1) / kShPartRows; }

// Rows of an L-phase wave's l-segment: the most (up to kShSegRows) that still give the batch kMinLWaves waves.
// A wave walks its rows one pair after another, so a small batch's L-phase takes as long as one segment; long
// segments re-read fewer halo rows (7 per segment). Segments of 4 rows walk 11 rows where those of 8 walk 15, but
// twice as many of them: only where 8 rows leave fewer waves than there are SIMDs (1 / 2 / 3 / 4 meshes of 200 x 1000,
// 400 waves each: 8 rows 19.2 / 21.1 / 22.1 / 24.2 us, 4 rows 18.3 / 20.6 / 22.0 / 29.1). us per step with 4 / 8 / 16 / 32 / 64
// rows: 250 x 100 14.4 / 15.9 / 18.8 / 23.9 / 30.8, 1000 x 200 21.1 / 22.2 / 24.7 / 30.9 / 38.4; with 8 / 16 / 32 / 64,
// simulations of 500 to 4000 radial points: 4 M points 95 / 92 / 92 / 99, 13 M 246 / 234 / 237 / 246, 48 M 762 / 697 /
// 705 / 724. The rule dates from a kernel of 4 waves per SIMD (the present one has 3): from about 4 M points on 16
// rows would be up to 4 % faster than its choice.
// `columns` counts, for every live simulation, its 64-position columns times its partials along l.
constexpr int64_t kMinLWaves = 4096, kMinLWaves8 = 1024;
int sh_segment_rows(int64_t columns) {
    int rows = kShSegRows;
    while (rows > 8 && columns * kShPartRows / rows < kMinLWaves) rows /= 2;
    return rows == 8 && columns * kShPartRows / 8 < kMinLWaves8 ? kShPartRows : rows;
}

int n_data_points(int N, int every) {
    if (every >= 1) return N / every + 1 + ((N % every) != 0 ? 1 : 0);
    return 2;
}

}  // namespace

struct tdse_ctx {
    int device = 0;
    int cus = 0;  // compute units
    hipStream_t stream = nullptr;
    Arena arena;
    std::string err;
    std::vector<ShHost> sh;
    std::vector<LineHost> line;
    std::vector<CylHost> cyl;
    ShSim* d_sh = nullptr;
    LineSim* d_line = nullptr;
    CylSim* d_cyl = nullptr;
    DevVec<int2> cyl_jobs, cyl_count_jobs;
    std::vector<Bucket> cyl_buckets;  // by (z and rho layout)
    double* d_cl = nullptr;
    double* d_clv = nullptr;  // c_l (l + 1): the velocity gauge's h1 coupling per l
    int* d_ctl = nullptr;     // [0] nonzero while the next replay of the current run follows (ADI run-ahead);
                              // [1] a tridiagonal line that was split has to be solved as one run
    DevVec<ShWave> waves;     // length-gauge simulations' waves first, then velocity-gauge ones
    int n_len_waves = 0;
    DevVec<int2> jobs;      // SH observations, and the step counts of all but the ADI simulations
    DevVec<int2> adi_jobs;  // the ADI simulations' step counts
    std::vector<Bucket> sh_buckets;
    std::vector<int> sh_order;  // sh_buckets by decreasing work
    std::vector<Bucket> sh_adi_buckets;  // AlternatingDirectionImplicit l-lines (slot, l) by (rows, chunks)
    DevVec<int2> adi_waves;              // AlternatingDirectionImplicit positions: (slot, first position of a wave)
    std::vector<Bucket> sh_adi_lbuckets;  // ADI position groups (slot, group) of the partition l-sweep, by rows
    hipStream_t side[3] = {nullptr, nullptr, nullptr};
    hipEvent_t ev_fork = nullptr, ev_join[3] = {nullptr, nullptr, nullptr};
    // every layout in one launch for each sweep (any_layouts): the buckets' lines, longest first
    bool any_sh = false, any_adi = false;
    DevVec<int2> any_lines, any_pairs, any_adi_lines, any_adi_groups;
    int any_threads = 0, any_pair_threads = 0, any_adi_threads = 0;
    size_t any_lds = 0, any_adi_lds = 0;
    bool any_has_pairs = false;  // some entries of any_lines are velocity odd l-pairs
    std::vector<Bucket> line_buckets;
    bool dirty = true;
    bool sh_norm_by_l = false;   // some live SH simulation reduces the norm in every l (L-phase instance)
    bool cyl_pending = false;    // a cylindrical simulation was added or uploaded: it starts from an exact state
    bool graph_cyl_pre = false;  // the captured step includes the cylindrical pre-sweep
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    hipGraph_t graph_k = nullptr;  // kGraphSteps steps in one graph (fewer launches for small batches)
    hipGraphExec_t exec_k = nullptr;
    hipEvent_t ev_start = nullptr, ev_stop = nullptr;
    double2* scratch = nullptr;  // this device's copy of `scratch` (tdse_tdma_batched_noalloc)
    double last_run_ms = 0.0;
    bool profiling = false;
    std::vector<hipEvent_t> ev_pool;
    size_t ev_used = 0;
    // (kind, start event index); kinds: SH L-phase, SH R-phase, Cyl z, Cyl rho, SH velocity-gauge h2
    // factors, SH velocity-gauge odd l-pair R-phase
    std::vector<std::pair<int, int>> ev_pairs;
    double prof_ms[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    int64_t prof_n[6] = {0, 0, 0, 0, 0, 0};
};

namespace {

int fail(tdse_ctx* ctx, int code, const std::string& msg) {
    if (ctx) ctx->err = msg;
    else g_lib_error = msg;
    return code;
}

#define HIP_TRY(ctx, expr)                                                                          \
    do {                                                                                            \
        hipError_t e_ = (expr);                                                                     \
        if (e_ != hipSuccess)                                                                       \
            return fail((ctx), TDSE_ERR_HIP, std::string(#expr) + ": " + hipGetErrorString(e_));    \
    } while (0)

template <class T>
int devvec_upload(tdse_ctx* ctx, DevVec<T>& v, const std::vector<T>& host) {
    if (host.size() > v.cap) {
        if (v.ptr) HIP_TRY(ctx, hipFree(v.ptr));
        v.cap = std::max<size_t>(host.size(), 2 * v.cap);
        HIP_TRY(ctx, hipMalloc(&v.ptr, v.cap * sizeof(T)));
    }
    v.count = host.size();
    if (!host.empty())
        HIP_TRY(ctx, hipMemcpyAsync(v.ptr, host.data(), host.size() * sizeof(T), hipMemcpyHostToDevice, ctx->stream));
    return TDSE_OK;
}

void drop_graph(tdse_ctx* ctx) {
    if (ctx->exec) (void)hipGraphExecDestroy(ctx->exec);
    if (ctx->graph) (void)hipGraphDestroy(ctx->graph);
    if (ctx->exec_k) (void)hipGraphExecDestroy(ctx->exec_k);
    if (ctx->graph_k) (void)hipGraphDestroy(ctx->graph_k);
    ctx->exec = nullptr;
    ctx->graph = nullptr;
    ctx->exec_k = nullptr;
    ctx->graph_k = nullptr;
}

size_t line_lds_bytes(int P);
size_t cn_lds_bytes(int M, int P, int form);
int cn_form(int M, int P);
size_t vpair_lds_bytes(int M, int P);
size_t adi_lds_bytes(int P);

// Whether the layouts of a set of lines share one launch per sweep (any_layouts): none past kAnyP threads, a batch of
// at most 24 M points (12 M with velocity-gauge pairs, counted as half their points, or ADI's three sweeps), and
// workgroups that lose little by it. What a shared launch saves are the other launches with their forks and joins, 10
// to 50 us a step; what it costs is occupancy: every workgroup takes the threads and the LDS of the deepest
// line, and the registers of 2 waves per SIMD. AnyCost adds up, over the workgroups, the share of a CU that each takes there
// beyond its share in its layout's own launch: CU-rounds lost. In the length gauge the waves past a line's threads
// leave at once and count half. One launch against a launch for each layout was faster in 170 batches while
// the loss was below about 3 rounds (length gauge), 0.4 per layout and 0.4 more (velocity gauge, whose chains have more
// launches each) and 13.5 (ADI, r-lines and l-groups together); a rule by points alone took the slower one by up to a
// factor of 2.5. us per step, one launch / one for each layout, and the rounds lost:
//   length-gauge simulations of 500 to 4000 radial points    4 M points   86 / 106 (0.8)    16 M  298 / 279 (4.5)
//   velocity-gauge ones                                      4 M         206 / 256 (2.7)     9 M  443 / 375 (8)
//   a 4000 x 50 mesh beside 250 x 50 ones, length gauge     50 of them    35 /  41 (2.4)    200    94 /  77 (9.8)
//   the same, velocity gauge                                10            58 /  76 (0.9)    200   303 / 144 (18)
//   the same, ADI                                           50            59 /  72 (6.4)    200   157 / 105 (24)
using Layouts = std::map<std::pair<int, int>, std::vector<int2>>;  // (rows, chunks) -> lines
constexpr int64_t kAnyPoints = int64_t(24) << 20;       // single lines only
constexpr int64_t kAnyPointsMore = int64_t(12) << 20;   // with velocity-gauge pairs, or ADI's three sweeps
constexpr double kAnyLost = 3.0, kAnyLostPairs = 0.4, kAnyLostAdi = 13.2;
bool any_layouts(const Layouts& lines, const Layouts& pairs, int64_t limit) {
    int64_t points = 0;
    for (const Layouts* m : {&lines, &pairs})
        for (auto& kv : *m) {
            if (kv.first.second > kAnyP) return false;
            points += (int64_t)kv.second.size() * kv.first.first * kv.first.second;
        }
    return points <= limit;
}
struct AnyCost {
    size_t lds;     // of the shared launch
    double waves;   // of its workgroups
    double lost = 0.0;
    static double share(size_t lds, double waves, int per_simd) {
        return std::max((double)lds / (160 << 10), waves / (4 * per_simd));
    }
    // count workgroups of a layout whose own launch has own_lds, own_waves and rows per thread M;
    // early: the part of the surplus waves' share that they give back by leaving
    void add(size_t count, size_t own_lds, double own_waves, int M, double early = 0.0) {
        const int per_simd = M <= 8 ? 4 : M == 10 ? 3 : 2;  // as launched (launch_rphase, launch_adi_lp)
        lost += (double)count * (share(lds, waves - early * (waves - own_waves), 2) - share(own_lds, own_waves, per_simd));
    }
};

// The single-launch tables of the split-operator and ADI simulations (longest lines first).
int build_any(tdse_ctx* ctx, const Layouts& lines, const Layouts (&vpairs)[2], const Layouts& fpairs,
              const Layouts& adi, const Layouts& adi_groups) {
    std::vector<int2> solve, pairs, al, ag;
    int rc;
    ctx->any_sh = lines.size() + fpairs.size() > 1 &&
                  any_layouts(lines, fpairs, fpairs.empty() ? kAnyPoints : kAnyPointsMore / 2);
    // one layout in each of ADI's sweeps: nothing to share
    ctx->any_adi = (adi.size() > 1 || adi_groups.size() > 1) && any_layouts(adi, adi_groups, kAnyPointsMore) &&
                   ctx->adi_waves.count == 0;
    ctx->any_threads = ctx->any_pair_threads = ctx->any_adi_threads = 0;
    ctx->any_lds = ctx->any_adi_lds = 0;
    ctx->any_has_pairs = false;
    for (auto& kv : fpairs) {
        ctx->any_threads = std::max(ctx->any_threads, 2 * kv.first.second);
        ctx->any_lds = std::max(ctx->any_lds, vpair_lds_bytes(kv.first.first, kv.first.second));
    }
    for (auto& kv : lines) {
        const int M = kv.first.first, P = kv.first.second;
        ctx->any_threads = std::max(ctx->any_threads, P);
        ctx->any_lds = std::max(ctx->any_lds, cn_lds_bytes(M, P, cn_form(M, P)));
    }
    if (ctx->any_sh) {
        AnyCost cost{ctx->any_lds, (double)ctx->any_threads / TDSE_WAVE};
        for (auto& kv : fpairs) {
            const int M = kv.first.first, P = kv.first.second;
            cost.add(kv.second.size(), vpair_lds_bytes(M, P), 2.0 * P / TDSE_WAVE, M);
        }
        for (auto& kv : lines) {
            const int M = kv.first.first, P = kv.first.second;
            cost.add(kv.second.size(), cn_lds_bytes(M, P, cn_form(M, P)), (double)P / TDSE_WAVE, M, fpairs.empty() ? 0.5 : 0.0);
        }
        const double most = fpairs.empty() ? kAnyLost : kAnyLostPairs * (1.0 + (double)lines.size());
        ctx->any_sh = cost.lost <= most * ctx->cus;
    }
    for (auto& kv : adi) {
        ctx->any_adi_threads = std::max(ctx->any_adi_threads, kv.first.second);
        ctx->any_adi_lds = std::max(ctx->any_adi_lds, adi_lds_bytes(kv.first.second));
    }
    if (ctx->any_adi) {
        AnyCost r{ctx->any_adi_lds, (double)ctx->any_adi_threads / TDSE_WAVE};
        for (auto& kv : adi) r.add(kv.second.size(), adi_lds_bytes(kv.first.second), (double)kv.first.second / TDSE_WAVE, kv.first.first);
        const size_t group_lds = adi_lds_bytes(kAdiChunks * kAdiLanes);
        AnyCost l{group_lds, (double)(kAdiChunks * kAdiLanes) / TDSE_WAVE};
        for (auto& kv : adi_groups) l.add(kv.second.size(), group_lds, l.waves, kv.first.first);
        ctx->any_adi = r.lost + l.lost <= kAnyLostAdi * ctx->cus;
    }
    if (ctx->any_sh) {
        for (auto it = fpairs.rbegin(); it != fpairs.rend(); ++it) {
            for (const int2& e : it->second) solve.push_back(make_int2(e.x, e.y | kAnyPair));
            ctx->any_has_pairs = true;
        }
        for (auto it = lines.rbegin(); it != lines.rend(); ++it) solve.insert(solve.end(), it->second.begin(), it->second.end());
        // up to kAnyP threads the odd l-pairs are solved with the lines: only the even ones are left
        for (auto it = vpairs[0].rbegin(); it != vpairs[0].rend(); ++it) {
            pairs.insert(pairs.end(), it->second.begin(), it->second.end());
            ctx->any_pair_threads = std::max(ctx->any_pair_threads, sh_vel_split(it->first.first) * it->first.second);
        }
    }
    if (ctx->any_adi) {
        for (auto it = adi.rbegin(); it != adi.rend(); ++it) al.insert(al.end(), it->second.begin(), it->second.end());
        for (auto it = adi_groups.rbegin(); it != adi_groups.rend(); ++it)
            ag.insert(ag.end(), it->second.begin(), it->second.end());
    }
    if ((rc = devvec_upload(ctx, ctx->any_lines, solve)) || (rc = devvec_upload(ctx, ctx->any_pairs, pairs)) ||
        (rc = devvec_upload(ctx, ctx->any_adi_lines, al)) || (rc = devvec_upload(ctx, ctx->any_adi_groups, ag)))
        return rc;
    HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));  // the host vectors end here
    return TDSE_OK;
}

// Rebuild the ragged work tables from the live simulations.
int rebuild_tables(tdse_ctx* ctx) {
    std::vector<ShWave> waves;
    std::vector<int2> jobs, ajobs;
    ctx->n_len_waves = -1;
    std::map<std::pair<int, int>, std::vector<int2>> shb, lnb;  // (rows, chunks [+ 4096 if complex steps])
    std::map<std::pair<bool, int>, std::vector<int>> lna;       // lines of any layout, (complex steps, method)
    std::map<std::pair<int, int>, std::vector<int2>> vpb[2];    // velocity l-pairs by parity, (rows, chunks)
    std::map<std::pair<int, int>, std::vector<int2>> fpb;       // velocity odd l-pairs solved in one workgroup
    std::map<std::pair<int, int>, std::vector<int2>> adb;       // ADI l-lines, (rows, chunks)
    std::vector<int2> adw;                                      // ADI position waves (Thomas l-sweep)
    std::map<std::pair<int, int>, std::vector<int2>> alb;       // ADI position groups (partition l-sweep), (rows, 0)
    ctx->sh_norm_by_l = false;
    int64_t columns = 0;
    for (const ShHost& h : ctx->sh)
        if (h.live) columns += (int64_t)(h.dev.npad / TDSE_WAVE) * sh_parts(h.dev.L);
    const int seg_parts = sh_segment_rows(columns) / kShPartRows;
    for (int pass = 0; pass < 2; ++pass)
    for (int s = 0; s < (int)ctx->sh.size(); ++s) {
        ShHost& h = ctx->sh[s];
        if (!h.live || (int)h.vel != pass) continue;
        if (pass == 1 && ctx->n_len_waves < 0) ctx->n_len_waves = (int)waves.size();
        h.wave_first = (int)waves.size();
        const int parts = sh_parts(h.dev.L);
        const int nseg = (parts + seg_parts - 1) / seg_parts;
        const int seg = (parts + nseg - 1) / nseg * kShPartRows;  // balanced, whole partials
        const int wpl = h.dev.npad / TDSE_WAVE;
        for (int lo = 0; lo < h.dev.L; lo += seg) {
            const int hi = std::min(h.dev.L, lo + seg);
            for (int w = 0; w < wpl; ++w) waves.push_back(ShWave{s, w * TDSE_WAVE, lo, hi});
        }
        h.wave_count = (int)waves.size() - h.wave_first;
        (h.adi ? ajobs : jobs).push_back(make_int2(s, -3));
        jobs.push_back(make_int2(s, -1));
        if (h.dev.norm_by_l) {
            jobs.push_back(make_int2(s, -2));
            ctx->sh_norm_by_l = true;
        }
        for (int b = 0; b < h.dev.n_basis; ++b) jobs.push_back(make_int2(s, b));
        if (h.adi) {
            for (int l = 0; l < h.dev.L; ++l) adb[{h.dev.m, h.dev.P}].push_back(make_int2(s, l));
            // l-direction: the partition solver where kAdiChunks chunks of at most 16 rows cover l_bound
            const int ml = sh_adi_lp_rows(h.dev.L);
            if (ml <= 16) {
                for (int gq = 0; gq < h.dev.npad / kAdiLanes; ++gq) alb[{ml, 0}].push_back(make_int2(s, gq));
            } else {
                for (int w = 0; w < wpl; ++w) adw.push_back(make_int2(s, w * TDSE_WAVE));
            }
            continue;
        }
        auto& v = shb[{h.dev.m, h.dev.P}];
        // velocity gauge: where two lines fit one workgroup (2 P <= 512) the odd l-pairs are
        // solved together with their h2 factors; the rows outside them stay single lines
        const bool fuse = h.vel && 2 * h.dev.P <= kMaxPairThreads;
        for (int l = 0; l < h.dev.L; ++l) {
            const bool in_odd_pair = (l & 1) ? (l + 1 < h.dev.L) : (l >= 1);
            if (!(fuse && in_odd_pair)) v.push_back(make_int2(s, l));
        }
        if (h.vel)
            for (int l = 0; l + 1 < h.dev.L; ++l) {
                if (fuse && (l & 1)) fpb[{h.dev.m, h.dev.P}].push_back(make_int2(s, l));
                else vpb[l & 1][{h.dev.m, h.dev.P}].push_back(make_int2(s, l));
            }
    }
    if (ctx->n_len_waves < 0) ctx->n_len_waves = (int)waves.size();
    int n_lines = 0;
    for (const LineHost& h : ctx->line) n_lines += h.live;
    // at most one line per CU: one launch for all layouts of a method (bucket M == 0)
    const bool any_layout = n_lines <= ctx->cus;
    for (int s = 0; s < (int)ctx->line.size(); ++s) {
        const LineHost& h = ctx->line[s];
        if (!h.live) continue;
        if (any_layout) lna[{h.complex_steps, h.dev.method}].push_back(s);
        else lnb[{h.dev.m, h.dev.P + (h.complex_steps ? 4096 : 0) + 8192 * h.dev.method}].push_back(make_int2(s, 0));
    }
    std::vector<int2> cjobs, ccount;
    std::map<std::array<int, 5>, std::pair<std::vector<int2>, std::vector<int2>>> cyb;  // (Mz, Pz, Mr, Cr, lanes)
    for (int s = 0; s < (int)ctx->cyl.size(); ++s) {
        const CylHost& h = ctx->cyl[s];
        if (!h.live) continue;
        const CylSim& C = h.dev;
        cjobs.push_back(make_int2(s, -1));
        cjobs.push_back(make_int2(s, -3));
        ccount.push_back(make_int2(s, -3));
        for (int b = 0; b < C.n_basis; ++b) cjobs.push_back(make_int2(s, b));
        auto& v = cyb[{C.Mz, C.Pz, C.Mr, C.Cr, C.lanes}];
        for (int q = 0; 2 * q < C.nr; ++q) v.first.push_back(make_int2(s, q));  // pairs of rho-lines
        for (int g = 0; g < C.n_groups; ++g) v.second.push_back(make_int2(s, g));
    }
    int rc;
    if ((rc = devvec_upload(ctx, ctx->waves, waves))) return rc;
    if ((rc = devvec_upload(ctx, ctx->jobs, jobs))) return rc;
    if ((rc = devvec_upload(ctx, ctx->adi_jobs, ajobs))) return rc;
    if ((rc = devvec_upload(ctx, ctx->cyl_jobs, cjobs))) return rc;
    if ((rc = devvec_upload(ctx, ctx->cyl_count_jobs, ccount))) return rc;
    auto fill = [&](std::vector<Bucket>& dst, std::map<std::pair<int, int>, std::vector<int2>>& src) -> int {
        for (auto& b : dst) free_bucket(b);
        dst.clear();
        for (auto& kv : src) {
            Bucket b;
            b.M = kv.first.first;
            b.P = kv.first.second % 4096;
            b.imag = (kv.first.second % 8192) >= 4096;
            b.method = kv.first.second / 8192;
            int r = devvec_upload(ctx, b.lines, kv.second);
            if (r) return r;
            dst.push_back(b);
        }
        return TDSE_OK;
    };
    for (auto& kv : fpb) shb[kv.first];  // a bucket for every layout with fused pairs, even without single lines
    if ((rc = fill(ctx->sh_buckets, shb))) return rc;
    if ((rc = fill(ctx->sh_adi_buckets, adb))) return rc;
    if ((rc = fill(ctx->sh_adi_lbuckets, alb))) return rc;
    if ((rc = devvec_upload(ctx, ctx->adi_waves, adw))) return rc;
    for (auto& b : ctx->sh_buckets) {
        for (int par = 0; par < 2; ++par) {
            auto it = vpb[par].find({b.M, b.P});
            if (it != vpb[par].end() && (rc = devvec_upload(ctx, b.vpairs[par], it->second))) return rc;
        }
        auto it = fpb.find({b.M, b.P});
        if (it != fpb.end() && (rc = devvec_upload(ctx, b.fpairs, it->second))) return rc;
    }
    if ((rc = build_any(ctx, shb, vpb, fpb, adb, alb))) return rc;
    if ((rc = fill(ctx->line_buckets, lnb))) return rc;
    for (auto& kv : lna) {
        ctx->line_buckets.emplace_back();
        Bucket& b = ctx->line_buckets.back();
        b.imag = kv.first.first;
        b.method = kv.first.second;
        // longest lines first; one layout keeps its own instance (fewer registers, exact block size)
        std::stable_sort(kv.second.begin(), kv.second.end(),
                         [&](int x, int y) { return ctx->line[x].dev.npad > ctx->line[y].dev.npad; });
        std::vector<int2> ids;
        bool one_layout = true;
        const LineSim& first = ctx->line[kv.second[0]].dev;
        for (int s : kv.second) {
            const LineSim& S = ctx->line[s].dev;
            ids.push_back(make_int2(s, 0));
            one_layout = one_layout && S.m == first.m && S.P == first.P;
            b.P = std::max(b.P, S.P);
            b.lds = std::max(b.lds, line_lds_bytes(S.P));
        }
        b.M = one_layout ? first.m : 0;
        if ((rc = devvec_upload(ctx, b.lines, ids))) return rc;
    }
    for (auto& b : ctx->cyl_buckets) free_bucket(b);
    ctx->cyl_buckets.clear();
    for (auto& kv : cyb) {
        ctx->cyl_buckets.emplace_back();
        Bucket& b = ctx->cyl_buckets.back();
        b.M = kv.first[0];
        b.P = kv.first[1];
        b.Mr = kv.first[2];
        b.Cr = kv.first[3];
        b.lanes = kv.first[4];
        if ((rc = devvec_upload(ctx, b.lines, kv.second.first)) || (rc = devvec_upload(ctx, b.rlines, kv.second.second)))
            return rc;
    }
    {
        std::vector<std::pair<double, int>> w;
        for (size_t i = 0; i < ctx->sh_buckets.size(); ++i) {
            // rows swept per step: the R-phase's lines, and the velocity-gauge h2 factors' rows
            // (two rows per pair, before and after the solve)
            const Bucket& b = ctx->sh_buckets[i];
            const double rows = (double)b.lines.count + 2.0 * (double)b.fpairs.count +
                                4.0 * (double)(b.vpairs[0].count + b.vpairs[1].count);
            w.push_back({-rows * b.P * b.M, (int)i});
        }
        std::sort(w.begin(), w.end());
        ctx->sh_order.clear();
        for (auto& pr : w) ctx->sh_order.push_back(pr.second);
    }
    HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
    drop_graph(ctx);
    ctx->dirty = false;
    return TDSE_OK;
}

hipEvent_t next_event(tdse_ctx* ctx) {
    if (ctx->ev_used == ctx->ev_pool.size()) {
        hipEvent_t e;
        (void)hipEventCreate(&e);
        ctx->ev_pool.push_back(e);
    }
    return ctx->ev_pool[ctx->ev_used++];
}

void prof_begin(tdse_ctx* ctx, int kind) {
    if (!ctx->profiling) return;
    ctx->ev_pairs.push_back({kind, (int)ctx->ev_used});
    (void)hipEventRecord(next_event(ctx), ctx->stream);
}
void prof_end(tdse_ctx* ctx) {
    if (!ctx->profiling) return;
    (void)hipEventRecord(next_event(ctx), ctx->stream);
}

// Form of a CN line kernel with M rows per thread and P threads: the
// explicit right-hand side for M >= 10; for M <= 8 the Cayley form, keeping
// the original rows in LDS when that fits the 64 KiB a workgroup gets by
// default, else re-reading them. Chosen from kernel-trace timings.
int cn_form(int M, int P) {
    if (M >= 10) return CN_EXPLICIT;
    return ((3 + M) * (size_t)P + kRedScratch) * sizeof(double2) <= 65536 ? CN_CAYLEY_LDS : CN_CAYLEY_MEM;
}
size_t cn_lds_bytes(int M, int P, int form) {
    return ((size_t)(form == CN_CAYLEY_LDS ? 3 + M : 3) * P + kRedScratch) * sizeof(double2);
}

// A job list as leading workgroups of a launch of `threads` per workgroup (none: no jobs ride there).
ShObs obs_of(const tdse_ctx* ctx, const DevVec<int2>& list, int threads, bool ride) {
    const int per = threads / TDSE_WAVE, nj = ride ? (int)list.count : 0;
    return ShObs{ctx->d_sh, list.ptr, nj, (nj + per - 1) / per, ctx->d_ctl};
}

// Launch shapes per rows-per-thread M (block size, minimum waves per EU).
template <int M, int MAXT, int WPE>
void launch_rphase(tdse_ctx* ctx, const Bucket& b, hipStream_t st, bool ride) {
    const int form = cn_form(M, b.P);
    const size_t lds = cn_lds_bytes(M, b.P, form);
    const ShObs obs = obs_of(ctx, ctx->jobs, b.P, ride);
    const dim3 grid((unsigned)(b.lines.count + obs.blocks)), block(b.P);
    if (form == CN_EXPLICIT)
        hipLaunchKernelGGL((k_sh_rphase<M, MAXT, WPE, (M >= 10 ? CN_EXPLICIT : CN_CAYLEY_MEM)>), grid, block, lds,
                           st, ctx->d_sh, b.lines.ptr, (int)b.lines.count, obs);
    else if (form == CN_CAYLEY_LDS)
        hipLaunchKernelGGL((k_sh_rphase<M, MAXT, WPE, (M >= 10 ? CN_EXPLICIT : CN_CAYLEY_LDS)>), grid, block, lds,
                           st, ctx->d_sh, b.lines.ptr, (int)b.lines.count, obs);
    else
        hipLaunchKernelGGL((k_sh_rphase<M, MAXT, WPE, (M >= 10 ? CN_EXPLICIT : CN_CAYLEY_MEM)>), grid, block, lds,
                           st, ctx->d_sh, b.lines.ptr, (int)b.lines.count, obs);
}

void dispatch_rphase(tdse_ctx* ctx, const Bucket& b, hipStream_t st, bool ride) {
    switch (b.M) {
        case 2: launch_rphase<2, 512, 4>(ctx, b, st, ride); break;
        case 4: launch_rphase<4, 512, 4>(ctx, b, st, ride); break;
        case 6: launch_rphase<6, 512, 4>(ctx, b, st, ride); break;
        case 8: launch_rphase<8, 512, 4>(ctx, b, st, ride); break;
        // radial lines past 4096 points: 512-thread workgroups of deep tiles
        case 10: b.P > 256 ? launch_rphase<10, 512, 1>(ctx, b, st, ride) : launch_rphase<10, 256, 3>(ctx, b, st, ride); break;
        case 12: b.P > 256 ? launch_rphase<12, 512, 1>(ctx, b, st, ride) : launch_rphase<12, 256, 2>(ctx, b, st, ride); break;
        case 14: b.P > 256 ? launch_rphase<14, 512, 1>(ctx, b, st, ride) : launch_rphase<14, 256, 2>(ctx, b, st, ride); break;
        default: b.P > 256 ? launch_rphase<16, 512, 1>(ctx, b, st, ride) : launch_rphase<16, 256, 1>(ctx, b, st, ride); break;
    }
}

size_t adi_lds_bytes(int P) { return (3 * (size_t)P + kRedScratch) * sizeof(double2); }

template <int M, int MAXT, int WPE, bool EXPL>
void launch_adi_r(tdse_ctx* ctx, const Bucket& b, hipStream_t st, bool ride) {
    const size_t lds = adi_lds_bytes(b.P);
    const ShObs obs = obs_of(ctx, EXPL ? ctx->jobs : ctx->adi_jobs, b.P, ride);
    hipLaunchKernelGGL((k_sh_adi_r<M, MAXT, WPE, EXPL>), dim3((unsigned)(b.lines.count + obs.blocks)), dim3(b.P), lds,
                       st, ctx->d_sh, b.lines.ptr, (int)b.lines.count, ctx->d_ctl, obs);
}

// the R-phase's launch shapes
template <bool EXPL>
void dispatch_adi_r(tdse_ctx* ctx, const Bucket& b, hipStream_t st, bool ride) {
    switch (b.M) {
        case 2: launch_adi_r<2, 512, 4, EXPL>(ctx, b, st, ride); break;
        case 4: launch_adi_r<4, 512, 4, EXPL>(ctx, b, st, ride); break;
        case 6: launch_adi_r<6, 512, 4, EXPL>(ctx, b, st, ride); break;
        case 8: launch_adi_r<8, 512, EXPL ? 4 : 3, EXPL>(ctx, b, st, ride); break;  // the run-ahead's registers
        case 10: b.P > 256 ? launch_adi_r<10, 512, 1, EXPL>(ctx, b, st, ride) : launch_adi_r<10, 256, 3, EXPL>(ctx, b, st, ride); break;
        case 12: b.P > 256 ? launch_adi_r<12, 512, 1, EXPL>(ctx, b, st, ride) : launch_adi_r<12, 256, 2, EXPL>(ctx, b, st, ride); break;
        case 14: b.P > 256 ? launch_adi_r<14, 512, 1, EXPL>(ctx, b, st, ride) : launch_adi_r<14, 256, 2, EXPL>(ctx, b, st, ride); break;
        default: b.P > 256 ? launch_adi_r<16, 512, 1, EXPL>(ctx, b, st, ride) : launch_adi_r<16, 256, 2, EXPL>(ctx, b, st, ride); break;
    }
}

template <int M>
void launch_adi_lp(tdse_ctx* ctx, const Bucket& b, hipStream_t st) {
    const size_t lds = (3 * (size_t)kAdiChunks * kAdiLanes + kRedScratch) * sizeof(double2);
    hipLaunchKernelGGL(k_sh_adi_lp<M>, dim3((unsigned)b.lines.count), dim3(kAdiChunks * kAdiLanes), lds, st,
                       ctx->d_sh, b.lines.ptr, (int)b.lines.count, ctx->d_cl);
}

void dispatch_adi_lp(tdse_ctx* ctx, const Bucket& b, hipStream_t st) {
    switch (b.M) {
        case 2: launch_adi_lp<2>(ctx, b, st); break;
        case 4: launch_adi_lp<4>(ctx, b, st); break;
        case 6: launch_adi_lp<6>(ctx, b, st); break;
        case 8: launch_adi_lp<8>(ctx, b, st); break;
        case 10: launch_adi_lp<10>(ctx, b, st); break;
        case 12: launch_adi_lp<12>(ctx, b, st); break;
        case 14: launch_adi_lp<14>(ctx, b, st); break;
        default: launch_adi_lp<16>(ctx, b, st); break;
    }
}

size_t vpair_lds_bytes(int M, int P) { return ((size_t)(3 + M - 2) * P * 2 + kRedScratch) * sizeof(double2); }

template <int M, int WPE>
void launch_rphase_vpair(tdse_ctx* ctx, const Bucket& b, hipStream_t st) {
    // the reduced system (3 P) and alpha_i of rows 0 .. M - 3 (M - 2 P) per line, two lines
    const size_t lds = vpair_lds_bytes(M, b.P);
    hipLaunchKernelGGL((k_sh_rphase_vpair<M, kMaxPairThreads, WPE>), dim3((unsigned)b.fpairs.count), dim3(2 * b.P),
                       lds, st, ctx->d_sh, b.fpairs.ptr, (int)b.fpairs.count, ctx->d_cl);
}

// waves per EU: the most that leave the two-line kernel without spills up to m = 14
void dispatch_rphase_vpair(tdse_ctx* ctx, const Bucket& b, hipStream_t st) {
    switch (b.M) {
        case 2: launch_rphase_vpair<2, 4>(ctx, b, st); break;
        case 4: launch_rphase_vpair<4, 4>(ctx, b, st); break;
        case 6: launch_rphase_vpair<6, 4>(ctx, b, st); break;
        case 8: launch_rphase_vpair<8, 3>(ctx, b, st); break;
        case 10: launch_rphase_vpair<10, 2>(ctx, b, st); break;
        case 12: launch_rphase_vpair<12, 2>(ctx, b, st); break;
        case 14: launch_rphase_vpair<14, 2>(ctx, b, st); break;
        default: launch_rphase_vpair<16, 1>(ctx, b, st); break;
    }
}

// Two threads per chunk (each with half its rows) where the halves keep an even row count and
// the workgroup stays within 512 threads: half the registers, twice the waves.
template <bool REV>
void dispatch_vphase(tdse_ctx* ctx, const Bucket& b, int par, hipStream_t st) {
    const DevVec<int2>& pairs = b.vpairs[par];
    const bool split = sh_vel_split(b.M) == 2 && 2 * b.P <= 512;
    const dim3 grid((unsigned)pairs.count), block((unsigned)(split ? 2 * b.P : b.P));
    auto args = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, grid, block, 0, st, ctx->d_sh, pairs.ptr, (int)pairs.count, ctx->d_cl);
    };
    switch (b.M) {
        case 2: args(k_sh_vphase<2, REV, 1>); break;
        case 4: args(k_sh_vphase<4, REV, 1>); break;
        case 6: args(k_sh_vphase<6, REV, 1>); break;
        case 8: split ? args(k_sh_vphase<8, REV, 2>) : args(k_sh_vphase<8, REV, 1>); break;
        case 10: args(k_sh_vphase<10, REV, 1>); break;
        case 12: split ? args(k_sh_vphase<12, REV, 2>) : args(k_sh_vphase<12, REV, 1>); break;
        case 14: args(k_sh_vphase<14, REV, 1>); break;
        default: split ? args(k_sh_vphase<16, REV, 2>) : args(k_sh_vphase<16, REV, 1>); break;
    }
}

size_t line_lds_bytes(int P) {
    return (3 * (size_t)P + kRedScratch) * sizeof(double2) + 64 * sizeof(double);
}

template <int M, bool IMAG, int METHOD>
void launch_line(tdse_ctx* ctx, const Bucket& b, int n_steps, hipStream_t st) {
    hipLaunchKernelGGL((k_line_steps<M, 512, IMAG, METHOD>), dim3((unsigned)b.lines.count), dim3(b.P),
                       line_lds_bytes(b.P), st, ctx->d_line, b.lines.ptr, (int)b.lines.count, n_steps);
}

// b.M == 0: lines of any layouts (k_line_steps_any), b.P the most threads and b.lds the most LDS of any of them
template <bool IMAG, int METHOD>
void dispatch_line_m(tdse_ctx* ctx, const Bucket& b, int n_steps, hipStream_t st) {
    switch (b.M) {
        case 0:
            hipLaunchKernelGGL((k_line_steps_any<512, IMAG, METHOD>), dim3((unsigned)b.lines.count), dim3(b.P), b.lds,
                               st, ctx->d_line, b.lines.ptr, (int)b.lines.count, n_steps);
            break;
        case 2: launch_line<2, IMAG, METHOD>(ctx, b, n_steps, st); break;
        case 4: launch_line<4, IMAG, METHOD>(ctx, b, n_steps, st); break;
        case 6: launch_line<6, IMAG, METHOD>(ctx, b, n_steps, st); break;
        case 8: launch_line<8, IMAG, METHOD>(ctx, b, n_steps, st); break;
        case 10: launch_line<10, IMAG, METHOD>(ctx, b, n_steps, st); break;
        case 12: launch_line<12, IMAG, METHOD>(ctx, b, n_steps, st); break;
        case 14: launch_line<14, IMAG, METHOD>(ctx, b, n_steps, st); break;
        default: launch_line<16, IMAG, METHOD>(ctx, b, n_steps, st); break;
    }
}

// complex time steps take the general instance (ADI only: the host rejects the
// split operator with complex steps)
void dispatch_line(tdse_ctx* ctx, const Bucket& b, int n_steps, hipStream_t st) {
    if (b.imag) dispatch_line_m<false, LINE_ADI>(ctx, b, n_steps, st);
    else if (b.method == LINE_SIO_LEN) dispatch_line_m<true, LINE_SIO_LEN>(ctx, b, n_steps, st);
    else if (b.method == LINE_SIO_VEL) dispatch_line_m<true, LINE_SIO_VEL>(ctx, b, n_steps, st);
    else dispatch_line_m<true, LINE_ADI>(ctx, b, n_steps, st);
}

// Run `launch(bucket, stream)` for every bucket over the context stream and the side streams (round robin),
// forked and joined by events: the buckets hold different simulations.
template <class F>
int fan_out(tdse_ctx* ctx, const std::vector<Bucket>& bs, F&& launch) {
    if (ctx->profiling || bs.size() < 2) {
        for (auto& b : bs) launch(b, ctx->stream);
        return TDSE_OK;
    }
    HIP_TRY(ctx, hipEventRecord(ctx->ev_fork, ctx->stream));
    for (int j = 0; j < kSideStreams; ++j) HIP_TRY(ctx, hipStreamWaitEvent(ctx->side[j], ctx->ev_fork, 0));
    for (size_t i = 0; i < bs.size(); ++i) {
        const int j = (int)(i % (kSideStreams + 1));
        launch(bs[i], j == 0 ? ctx->stream : ctx->side[j - 1]);
    }
    for (int j = 0; j < kSideStreams; ++j) {
        HIP_TRY(ctx, hipEventRecord(ctx->ev_join[j], ctx->side[j]));
        HIP_TRY(ctx, hipStreamWaitEvent(ctx->stream, ctx->ev_join[j], 0));
    }
    return TDSE_OK;
}

// The cylindrical observation jobs as leading workgroups of a launch of `threads` per workgroup.
CylJobs cyl_jobs_of(const tdse_ctx* ctx, const DevVec<int2>& list, int threads, bool ride) {
    const int per = threads / TDSE_WAVE, nj = ride ? (int)list.count : 0;
    return CylJobs{ctx->d_cyl, list.ptr, nj, (nj + per - 1) / per};
}

// The z-sweep solves two rho-lines per workgroup (2 Pz threads), explicit form
// (with two lines per workgroup the Cayley forms measured slower: re-reading the
// rows 0.44 ms, keeping them in LDS 0.64 ms per sweep against 0.40 ms).
template <int M, int MAXT, int WPE>
void launch_cyl_z(tdse_ctx* ctx, const Bucket& b, hipStream_t st, bool ride) {
    const size_t lds = cn_lds_bytes(M, 2 * b.P, CN_EXPLICIT);
    const CylJobs jobs = cyl_jobs_of(ctx, ctx->cyl_jobs, 2 * b.P, ride);
    hipLaunchKernelGGL((k_cyl_z<M, MAXT, WPE, CN_EXPLICIT>), dim3((unsigned)(b.lines.count + jobs.blocks)),
                       dim3(2 * b.P), lds, st, ctx->d_cyl, b.lines.ptr, (int)b.lines.count, jobs);
}

void dispatch_cyl_z(tdse_ctx* ctx, const Bucket& b, hipStream_t st, bool ride) {
    switch (b.M) {
        case 2: launch_cyl_z<2, 1024, 4>(ctx, b, st, ride); break;
        case 4: launch_cyl_z<4, 1024, 4>(ctx, b, st, ride); break;
        case 6: launch_cyl_z<6, 1024, 4>(ctx, b, st, ride); break;
        case 8: launch_cyl_z<8, 1024, 4>(ctx, b, st, ride); break;
        case 10: launch_cyl_z<10, 512, 3>(ctx, b, st, ride); break;
        case 12: launch_cyl_z<12, 512, 2>(ctx, b, st, ride); break;
        case 14: launch_cyl_z<14, 512, 2>(ctx, b, st, ride); break;
        default: launch_cyl_z<16, 512, 2>(ctx, b, st, ride); break;
    }
}

template <int M, int LANES, int MAXT, int WPE>
void launch_cyl_rho(tdse_ctx* ctx, const Bucket& b, hipStream_t st, int mode, bool ride) {
    const CylJobs jobs = cyl_jobs_of(ctx, ctx->cyl_count_jobs, b.Cr * LANES, ride);
    const size_t lds = cyl_rho_lds_bytes(M, LANES, b.Cr);
    const dim3 grid((unsigned)(b.rlines.count + jobs.blocks)), block((unsigned)(b.Cr * LANES));
    if (mode == CYL_PRE)
        hipLaunchKernelGGL((k_cyl_rho<M, LANES, CYL_PRE, MAXT, WPE>), grid, block, lds, st, ctx->d_cyl,
                           b.rlines.ptr, (int)b.rlines.count, jobs);
    else
        hipLaunchKernelGGL((k_cyl_rho<M, LANES, CYL_MAIN, MAXT, WPE>), grid, block, lds, st, ctx->d_cyl,
                           b.rlines.ptr, (int)b.rlines.count, jobs);
}

// rho-sweep shapes (rows, lines per workgroup, block limit, minimum waves per
// EU); the layout chooser of the host package picks one of these.
void dispatch_cyl_rho(tdse_ctx* ctx, const Bucket& b, hipStream_t st, int mode, bool ride) {
    if (b.Mr == 4 && b.lanes == 4) launch_cyl_rho<4, 4, 1024, 4>(ctx, b, st, mode, ride);
    else if (b.Mr == 8 && b.lanes == 4) launch_cyl_rho<8, 4, 512, 4>(ctx, b, st, mode, ride);
    else if (b.Mr == 4 && b.lanes == 8) launch_cyl_rho<4, 8, 1024, 4>(ctx, b, st, mode, ride);
    else if (b.Mr == 8 && b.lanes == 8) launch_cyl_rho<8, 8, 1024, 4>(ctx, b, st, mode, ride);
    else launch_cyl_rho<16, 4, 512, 2>(ctx, b, st, mode, ride);
}

// Reduce the pending observations of the cylindrical simulations.
void cyl_observe(tdse_ctx* ctx) {
    const CylJobs jobs = cyl_jobs_of(ctx, ctx->cyl_jobs, 256, true);
    hipLaunchKernelGGL(k_cyl_observe, dim3(jobs.blocks), dim3(256), 0, ctx->stream, jobs);
}

// Launch one full step of every simulation kind onto the context stream.
// cyl_pre: include the cylindrical pre-sweep (needed while any cylindrical
// simulation may start a step from an exact state).
int launch_step(tdse_ctx* ctx, bool cyl_pre) {
    const int nw = (int)ctx->waves.count;
    if (nw > 0) {
        prof_begin(ctx, 0);
        // the instance that reduces the norm in every l needs more registers: only when asked for
        const int nl = ctx->n_len_waves, nv = nw - nl;
        if (nl > 0) {
            auto lphase = ctx->sh_norm_by_l ? k_sh_lphase<true, false> : k_sh_lphase<false, false>;
            hipLaunchKernelGGL(lphase, dim3((nl * TDSE_WAVE + 255) / 256), dim3(256), 0, ctx->stream, ctx->d_sh,
                               ctx->waves.ptr, nl, ctx->d_cl, 0, ctx->d_sh);
        }
        if (nv > 0) {
            auto lphase = ctx->sh_norm_by_l ? k_sh_lphase<true, true> : k_sh_lphase<false, true>;
            hipLaunchKernelGGL(lphase, dim3((nv * TDSE_WAVE + 255) / 256), dim3(256), 0, ctx->stream, ctx->d_sh,
                               ctx->waves.ptr + nl, nv, ctx->d_clv, 0, ctx->d_sh);
        }
        prof_end(ctx);
        // The observables read only what the L-phase wrote (partials, snapshot rows), which nothing
        // else touches before the next replay: a few of them ride in the next launch (the smallest
        // R-phase bucket, or the first explicit ADI sweep), many get a launch beside the R-phase.
        const int nj = (int)ctx->jobs.count;
        const bool ride = nj <= kMaxRidingJobs;
        auto observe = [&](hipStream_t st) {
            if (ride) return;
            const ShObs obs = obs_of(ctx, ctx->jobs, 256, true);
            hipLaunchKernelGGL(k_sh_observe, dim3(obs.blocks), dim3(256), 0, st, obs);
        };
        const Bucket* rider = ctx->sh_order.empty() ? nullptr : &ctx->sh_buckets[ctx->sh_order.back()];
        // One bucket's chain: velocity-gauge h2 factors of its even, then odd l-pairs
        // (before the CN solve), the R-phase, the factors in reverse (after it). The
        // chains of different buckets touch different simulations.
        auto chain = [&](const Bucket& b, hipStream_t st) {
            for (int par = 0; par < 2; ++par)
                if (b.vpairs[par].count) {
                    prof_begin(ctx, 4);
                    dispatch_vphase<false>(ctx, b, par, st);
                    prof_end(ctx);
                }
            if (b.lines.count) {
                prof_begin(ctx, 1);
                dispatch_rphase(ctx, b, st, ride && &b == rider);
                prof_end(ctx);
            }
            if (b.fpairs.count) {
                prof_begin(ctx, 5);
                dispatch_rphase_vpair(ctx, b, st);
                prof_end(ctx);
            }
            for (int par = 1; par >= 0; --par)
                if (b.vpairs[par].count) {
                    prof_begin(ctx, 4);
                    dispatch_vphase<true>(ctx, b, par, st);
                    prof_end(ctx);
                }
        };
        if (ctx->any_sh && !ctx->profiling) {
            observe(ctx->stream);
            auto vphase = [&](auto kernel) {
                if (!ctx->any_pairs.count) return;
                hipLaunchKernelGGL(kernel, dim3((unsigned)ctx->any_pairs.count), dim3(ctx->any_pair_threads), 0,
                                   ctx->stream, ctx->d_sh, ctx->any_pairs.ptr, (int)ctx->any_pairs.count, ctx->d_cl);
            };
            const ShObs obs = obs_of(ctx, ctx->jobs, ctx->any_threads, ride);
            auto solve = [&](auto kernel) {
                hipLaunchKernelGGL(kernel, dim3((unsigned)(ctx->any_lines.count + obs.blocks)), dim3(ctx->any_threads),
                                   ctx->any_lds, ctx->stream, ctx->d_sh, ctx->any_lines.ptr,
                                   (int)ctx->any_lines.count, ctx->d_cl, obs);
            };
            vphase(k_sh_vphase_any<false>);
            if (ctx->any_has_pairs) solve(k_sh_solve_any<true>);
            else solve(k_sh_solve_any<false>);
            vphase(k_sh_vphase_any<true>);
        } else if (ctx->profiling || ctx->sh_buckets.size() < 2) {
            observe(ctx->stream);
            for (auto& b : ctx->sh_buckets) chain(b, ctx->stream);
        } else {
            // independent buckets run concurrently (largest first, round robin
            // over the context stream and the side streams) so that small
            // buckets fill the tails of large ones; fork and join by events
            HIP_TRY(ctx, hipEventRecord(ctx->ev_fork, ctx->stream));
            for (int j = 0; j < kSideStreams; ++j) HIP_TRY(ctx, hipStreamWaitEvent(ctx->side[j], ctx->ev_fork, 0));
            // the observables on the last side stream, which the round robin leaves the least work
            observe(ctx->side[kSideStreams - 1]);
            for (size_t i = 0; i < ctx->sh_order.size(); ++i) {
                const int j = (int)(i % (kSideStreams + 1));
                chain(ctx->sh_buckets[ctx->sh_order[i]], j == 0 ? ctx->stream : ctx->side[j - 1]);
            }
            for (int j = 0; j < kSideStreams; ++j) {
                HIP_TRY(ctx, hipEventRecord(ctx->ev_join[j], ctx->side[j]));
                HIP_TRY(ctx, hipStreamWaitEvent(ctx->stream, ctx->ev_join[j], 0));
            }
        }
        // AlternatingDirectionImplicit simulations: explicit H0, the l-direction factor, implicit H0.
        // Within each of the three sweeps the buckets are independent: they run concurrently
        // over the context stream and the side streams (fork and join by events), and each
        // sweep starts after the whole previous one.
        if (ctx->any_adi && !ctx->profiling) {
            const int nl = (int)ctx->any_adi_lines.count, ng = (int)ctx->any_adi_groups.count;
            const dim3 threads(ctx->any_adi_threads);
            const ShObs obs = obs_of(ctx, ctx->jobs, ctx->any_adi_threads, ride && !rider);
            const ShObs counts = obs_of(ctx, ctx->adi_jobs, ctx->any_adi_threads, true);
            hipLaunchKernelGGL(k_sh_adi_r_any<true>, dim3(nl + obs.blocks), threads,
                               ctx->any_adi_lds, ctx->stream,
                               ctx->d_sh, ctx->any_adi_lines.ptr, nl, ctx->d_ctl, obs);
            hipLaunchKernelGGL(k_sh_adi_lp_any, dim3(ng), dim3(kAdiChunks * kAdiLanes),
                               (3 * (size_t)kAdiChunks * kAdiLanes + kRedScratch) * sizeof(double2), ctx->stream,
                               ctx->d_sh, ctx->any_adi_groups.ptr, ng, ctx->d_cl);
            hipLaunchKernelGGL(k_sh_adi_r_any<false>, dim3(nl + counts.blocks), threads, ctx->any_adi_lds, ctx->stream,
                               ctx->d_sh, ctx->any_adi_lines.ptr, nl, ctx->d_ctl, counts);
        } else if (!ctx->sh_adi_buckets.empty()) {
            int rc;
            const Bucket* first = rider ? nullptr : &ctx->sh_adi_buckets[0];
            if ((rc = fan_out(ctx, ctx->sh_adi_buckets, [&](const Bucket& b, hipStream_t st) {
                    dispatch_adi_r<true>(ctx, b, st, ride && &b == first);
                })))
                return rc;
            if ((rc = fan_out(ctx, ctx->sh_adi_lbuckets, [&](const Bucket& b, hipStream_t st) { dispatch_adi_lp(ctx, b, st); })))
                return rc;
            const int na = (int)ctx->adi_waves.count;
            if (na > 0)
                hipLaunchKernelGGL(k_sh_adi_l, dim3((na * TDSE_WAVE + 255) / 256), dim3(256), 0, ctx->stream,
                                   ctx->d_sh, ctx->adi_waves.ptr, na, ctx->d_cl);
            if ((rc = fan_out(ctx, ctx->sh_adi_buckets, [&](const Bucket& b, hipStream_t st) {
                    dispatch_adi_r<false>(ctx, b, st, &b == &ctx->sh_adi_buckets[0]);
                })))
                return rc;
        }
    }
    if (int rc = fan_out(ctx, ctx->line_buckets, [&](const Bucket& b, hipStream_t st) { dispatch_line(ctx, b, 1, st); }))
        return rc;
    if (!ctx->cyl_buckets.empty()) {
        if (cyl_pre) {
            for (auto& b : ctx->cyl_buckets) dispatch_cyl_rho(ctx, b, ctx->stream, CYL_PRE, false);
            cyl_observe(ctx);
        }
        // one bucket's chain; the buckets hold different simulations. The jobs of all of them ride with the
        // first z-sweep (S.step is then still the same for every sweep) and the last rho-sweep.
        auto chain = [&](const Bucket& b, hipStream_t st) {
            prof_begin(ctx, 2);
            dispatch_cyl_z(ctx, b, st, &b == &ctx->cyl_buckets[0]);
            prof_end(ctx);
            prof_begin(ctx, 3);
            dispatch_cyl_rho(ctx, b, st, CYL_MAIN, &b == &ctx->cyl_buckets.back());
            prof_end(ctx);
        };
        for (auto& b : ctx->cyl_buckets) chain(b, ctx->stream);
    }
    HIP_TRY(ctx, hipGetLastError());
    return TDSE_OK;
}

// Capture `steps` consecutive steps into one graph.
int capture_steps(tdse_ctx* ctx, bool cyl_pre, int steps, hipGraph_t* graph, hipGraphExec_t* exec) {
    HIP_TRY(ctx, hipStreamBeginCapture(ctx->stream, hipStreamCaptureModeThreadLocal));
    int rc = 0;
    for (int i = 0; i < steps && !rc; ++i) rc = launch_step(ctx, cyl_pre);
    hipGraph_t g = nullptr;
    hipError_t e = hipStreamEndCapture(ctx->stream, &g);
    if (rc) {
        if (g) (void)hipGraphDestroy(g);
        return rc;
    }
    if (e != hipSuccess) return fail(ctx, TDSE_ERR_HIP, std::string("hipStreamEndCapture: ") + hipGetErrorString(e));
    *graph = g;
    HIP_TRY(ctx, hipGraphInstantiate(exec, g, nullptr, nullptr, 0));
    return TDSE_OK;
}

// The one-step graph and the kGraphSteps-step graph of the current tables.
int ensure_graph(tdse_ctx* ctx, bool cyl_pre) {
    if (ctx->exec && (kGraphSteps <= 1 || ctx->exec_k) && ctx->graph_cyl_pre == cyl_pre) return TDSE_OK;
    drop_graph(ctx);
    ctx->graph_cyl_pre = cyl_pre;
    int rc = capture_steps(ctx, cyl_pre, 1, &ctx->graph, &ctx->exec);
    if (!rc && kGraphSteps > 1) rc = capture_steps(ctx, cyl_pre, kGraphSteps, &ctx->graph_k, &ctx->exec_k);
    return rc;
}

template <class T>
int copy_to_device(tdse_ctx* ctx, std::vector<void*>& blocks, const T* host, size_t count, T** out) {
    const size_t bytes = std::max<size_t>(count, 1) * sizeof(T);
    void* p = ctx->arena.alloc(bytes);
    if (!p) return fail(ctx, TDSE_ERR_NOMEM, "device pool exhausted");
    blocks.push_back(p);
    if (host && count) HIP_TRY(ctx, hipMemcpyAsync(p, host, count * sizeof(T), hipMemcpyHostToDevice, ctx->stream));
    else HIP_TRY(ctx, hipMemsetAsync(p, 0, bytes, ctx->stream));
    *out = static_cast<T*>(p);
    return TDSE_OK;
}

// Plain streaming copy: one complex128 read and one write per element, the
// grid covering the buffer once (one element per thread up to 2^28 elements).
// On MI355X this form measured 6.2 TB/s for 1 GiB each way; a grid-stride
// loop over 8192 workgroups reached 4.5 TB/s.
__global__ void __launch_bounds__(256) k_stream_copy(const double2* __restrict__ src, double2* __restrict__ dst,
                                                     size_t n) {
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) st2(dst, i, ld2(src, i));
}

// Scratch of the allocation-free Thomas entry point: the primed super-diagonal
// of up to kNoAllocPoints unknowns, then kNoAllocSystems int64 offsets and as
// many int64 lengths (33 MiB in all). Each device holds its own copy until the
// process ends. In host code the name `scratch` is only a host-side stand-in:
// kernels and copies use the device address that hipGetSymbolAddress returns
// for the current device (device_scratch), never the name itself.
constexpr int64_t kNoAllocPoints = int64_t(1) << 21;
constexpr int64_t kNoAllocSystems = int64_t(1) << 16;
constexpr int kMaxDevices = 64;
static __device__ __align__(256) double2 scratch[kNoAllocPoints + kNoAllocSystems];

std::mutex g_scratch_mu;
double2* g_scratch_ptr[kMaxDevices] = {};

// Device address of `scratch` on `device` (which must be current), looked up
// once per device. Returns nullptr with *err set on failure.
double2* device_scratch(int device, hipError_t* err) {
    *err = hipSuccess;
    if (device < 0 || device >= kMaxDevices) {
        *err = hipErrorInvalidDevice;
        return nullptr;
    }
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_ptr[device]) {
        double2* p = nullptr;
        *err = hipGetSymbolAddress(reinterpret_cast<void**>(&p), HIP_SYMBOL(scratch));
        if (*err != hipSuccess) return nullptr;
        g_scratch_ptr[device] = p;
    }
    return g_scratch_ptr[device];
}

// Thomas solves of n_systems lines (lengths on the host and, as len, on the device): by one thread each
// (tdma_by_threads) or by waves. A line then gets one wave for
// every kTdmaSpan rows, of which those find work whose rows hold a restart (k_tdma_lines); the span
// grows where that would be more than kTdmaWaves workgroups. A second launch redoes every line as one run if
// a split line met a value that is not finite. in_place: x overlaps an input, which a second launch would find
// overwritten and another wave's search for restarts may: lines are then not split.
constexpr int64_t kTdmaSpan = 64, kTdmaWaves = int64_t(1) << 20;
hipError_t launch_tdma(tdse_ctx* ctx, const double2* a, const double2* b, const double2* c, const double2* d,
                       double2* x, double2* cp, const int64_t* off, const int64_t* len, const int64_t* lengths,
                       int64_t n_systems, bool in_place) {
    int64_t longest = 1, rows = 0;
    for (int64_t i = 0; i < n_systems; ++i) {
        longest = std::max(longest, lengths[i]);
        rows += lengths[i];
    }
    if (tdma_by_threads(n_systems, rows, longest)) {
        hipLaunchKernelGGL(k_tdma_threads, dim3((unsigned)((n_systems + TDSE_WAVE - 1) / TDSE_WAVE)), dim3(TDSE_WAVE), 0,
                           ctx->stream, a, b, c, d, x, cp, off, len, n_systems);
        return hipGetLastError();
    }
    const int64_t most = std::max<int64_t>(1, kTdmaWaves / n_systems);  // waves per line
    const int64_t span = in_place ? longest : std::max(kTdmaSpan, (longest + most - 1) / most);
    const int64_t per_line = (longest + span - 1) / span;
    int* redo = ctx->d_ctl + 1;
    hipError_t e = hipSuccess;
    if (per_line > 1) e = hipMemsetD32Async(reinterpret_cast<hipDeviceptr_t>(redo), 0, 1, ctx->stream);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_tdma_lines, dim3((unsigned)(n_systems * per_line)), dim3(TDSE_WAVE), 0, ctx->stream, a, b, c, d,
                       x, cp, off, len, n_systems, span, per_line, 0, redo);
    e = hipGetLastError();
    if (e != hipSuccess || per_line == 1) return e;
    hipLaunchKernelGGL(k_tdma_lines, dim3((unsigned)n_systems), dim3(TDSE_WAVE), 0, ctx->stream, a, b, c, d, x, cp, off,
                       len, n_systems, longest, int64_t(1), 1, redo);
    return hipGetLastError();
}

// A wavefunction between natural order and device positions: element (row, j) of an SH or Line g (n points per
// row, chunk layout P x m), or (jz, r) of a cylinder (cyl_at), rows row0 .. row0 + rows - 1. One thread per
// natural element, the natural side unit-stride. The host's own reordering (a NumPy gather and scatter over the padded
// copy) took 0.2 s for 15 M points, more than a third of a 2000-step run of them.
// After them, one thread per padding position of `pads` (null: none) writes its zero: the zero couplings of
// padding rows keep zeros, but not against a state that held a NaN or an infinity (0 * NaN), which
// the solves carry into every padding row that shares a line with it.
struct NaturalMap {
    int n, P, m, npad;  // points per natural row; chunk layout and padded length of the permuted index
    int rows;           // natural rows
    int rpad;           // cylinder: padded rho rows; else 0. The row index (z), not the column (rho), is then permuted
    __device__ int position(int j) const { return (j % m) * P + j / m; }
    __host__ __device__ int64_t padding() const {
        return rpad ? (int64_t)rpad * npad - (int64_t)rows * n : (int64_t)rows * (npad - n);
    }
    // Device element of padding position q < padding(): the indices past the end of the permuted index, then a
    // cylinder's rho rows past the last for the rest.
    __device__ size_t padding_at(int64_t q) const {
        const int over = npad - (rpad ? rows : n);
        if (!rpad) return (size_t)(q / over) * npad + position(n + (int)(q % over));
        const int64_t first = (int64_t)rpad * over;
        if (q < first) return cyl_at((int)(q / over), position(rows + (int)(q % over)), npad);
        return cyl_at(n + (int)((q - first) / rows), position((int)((q - first) % rows)), npad);
    }
};
struct PaddedStates {
    double2 *a = nullptr, *b = nullptr;
};
template <bool TO_NATURAL>
__global__ void __launch_bounds__(256) k_natural(double2* __restrict__ g, double2* __restrict__ nat, NaturalMap map,
                                                 int64_t row0, int64_t rows, PaddedStates pads) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= rows * map.n) {
        const int64_t q = i - rows * map.n;
        if (TO_NATURAL || q >= map.padding()) return;
        const size_t at = map.padding_at(q);
        if (pads.a) st2(pads.a, at, cmk(0.0, 0.0));
        if (pads.b) st2(pads.b, at, cmk(0.0, 0.0));
        return;
    }
    const int64_t row = row0 + i / map.n;
    const int col = (int)(i % map.n);
    const int p = map.position(map.rpad ? (int)row : col);
    const size_t at = map.rpad ? cyl_at(col, p, map.npad) : (size_t)row * map.npad + p;
    if (TO_NATURAL) st2(nat, (size_t)i, ld2(g, at));
    else st2(g, at, ld2(nat, (size_t)i));
}

// Move a whole wavefunction between the host (natural order) and the device through a staging block of the pool:
// all rows at once, or half, a quarter, ... of them, down to kStageBytes; below that, a block of that size which the
// context keeps past its pool. Upload and download of 2000 x 1000 points (32 MB): 3.2 ms with room, 3.3 with a
// full pool (79.9 row by row).
constexpr size_t kStageBytes = size_t(16) << 20;
template <bool TO_HOST>
int move_natural(tdse_ctx* ctx, double2* g, const NaturalMap& map, double2* host, const PaddedStates pads = {}) {
    const int64_t rows = map.rows;
    const size_t row_bytes = (size_t)map.n * sizeof(double2);
    int64_t chunk = rows;
    void* stage = nullptr;
    while (!(stage = ctx->arena.alloc((size_t)chunk * row_bytes)) && (size_t)chunk * row_bytes > kStageBytes)
        chunk = (chunk + 1) / 2;
    const bool pooled = stage;
    bool own = false;
    if (!pooled) {
        chunk = std::min(rows, std::max<int64_t>(1, (int64_t)(kStageBytes / row_bytes)));
        stage = ctx->arena.beyond;
        own = !stage;
        if (own) HIP_TRY(ctx, hipMalloc(&stage, (size_t)chunk * row_bytes));
    }
    double2* nat = static_cast<double2*>(stage);
    hipError_t e = hipSuccess;
    for (int64_t r = 0; r < rows && e == hipSuccess; r += chunk) {
        const int64_t k = std::min(chunk, rows - r), count = k * map.n;
        const PaddedStates clear = r + k == rows ? pads : PaddedStates{};  // with the last rows
        const dim3 grid((unsigned)((count + (clear.a ? map.padding() : 0) + 255) / 256));
        if (!TO_HOST)
            e = hipMemcpyAsync(nat, host + r * map.n, (size_t)k * row_bytes, hipMemcpyHostToDevice, ctx->stream);
        if (e == hipSuccess) {
            hipLaunchKernelGGL(k_natural<TO_HOST>, grid, dim3(256), 0, ctx->stream, g, nat, map, r, k, clear);
            e = hipGetLastError();
        }
        if (TO_HOST && e == hipSuccess)
            e = hipMemcpyAsync(host + r * map.n, nat, (size_t)k * row_bytes, hipMemcpyDeviceToHost, ctx->stream);
        // the staging block is used again, and the host buffer is the caller's
        if (e == hipSuccess) e = hipStreamSynchronize(ctx->stream);
    }
    if (e != hipSuccess) (void)hipStreamSynchronize(ctx->stream);
    if (own) (void)hipFree(stage);
    if (pooled) ctx->arena.dealloc(stage);
    return e == hipSuccess ? TDSE_OK : fail(ctx, TDSE_ERR_HIP, std::string("wavefunction copy: ") + hipGetErrorString(e));
}

// The live simulation's map; false for a bad kind or slot.
bool natural_of(const tdse_ctx* ctx, int32_t kind, int32_t slot, NaturalMap* map) {
    if (slot < 0) return false;
    if (kind == 0 && slot < (int)ctx->sh.size() && ctx->sh[slot].live) {
        const ShSim& S = ctx->sh[slot].dev;
        *map = NaturalMap{S.n, S.P, S.m, S.npad, S.L, 0};
        return true;
    }
    if (kind == 1 && slot < (int)ctx->line.size() && ctx->line[slot].live) {
        const LineSim& S = ctx->line[slot].dev;
        *map = NaturalMap{S.n, S.P, S.m, S.npad, 1, 0};
        return true;
    }
    if (kind == 2 && slot < (int)ctx->cyl.size() && ctx->cyl[slot].live) {
        const CylSim& S = ctx->cyl[slot].dev;
        *map = NaturalMap{S.nr, S.Pz, S.Mz, S.npz, S.nz, S.nrpad};
        return true;
    }
    return false;
}

void free_blocks(tdse_ctx* ctx, std::vector<void*>& blocks) {
    for (void* p : blocks) ctx->arena.dealloc(p);
    blocks.clear();
}

}  // namespace

// ====================================================================== C ABI

extern "C" {

int tdse_abi_version(void) { return kAbiVersion; }

const char* tdse_last_error(const tdse_ctx* ctx) { return ctx ? ctx->err.c_str() : g_lib_error.c_str(); }

int tdse_ctx_create(int device, size_t pool_bytes, tdse_ctx** out) {
    if (!out) return fail(nullptr, TDSE_ERR_ARG, "out is NULL");
    *out = nullptr;
    int count = 0;
    if (hipGetDeviceCount(&count) != hipSuccess || count == 0)
        return fail(nullptr, TDSE_ERR_HIP, "no HIP device available");
    if (device < 0 || device >= count) return fail(nullptr, TDSE_ERR_ARG, "device index out of range");
    if (hipSetDevice(device) != hipSuccess) return fail(nullptr, TDSE_ERR_HIP, "hipSetDevice failed");
    tdse_ctx* ctx = new tdse_ctx();
    ctx->device = device;
    if (hipDeviceGetAttribute(&ctx->cus, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess) ctx->cus = 0;
    if (hipStreamCreateWithFlags(&ctx->stream, hipStreamNonBlocking) != hipSuccess) {
        delete ctx;
        return fail(nullptr, TDSE_ERR_HIP, "hipStreamCreate failed");
    }
    if (!ctx->arena.init(pool_bytes, kStageBytes)) {
        (void)hipStreamDestroy(ctx->stream);
        delete ctx;
        return fail(nullptr, TDSE_ERR_NOMEM, "could not reserve the device memory pool");
    }
    std::vector<double> cl(kMaxL), clv(kMaxL);
    for (int l = 0; l < kMaxL; ++l) {
        cl[l] = (l + 1.0) / std::sqrt((2.0 * l + 1.0) * (2.0 * l + 3.0));
        clv[l] = cl[l] * (l + 1.0);
    }
    bool ok = hipMalloc(&ctx->d_cl, kMaxL * sizeof(double)) == hipSuccess &&
              hipMemcpy(ctx->d_cl, cl.data(), kMaxL * sizeof(double), hipMemcpyHostToDevice) == hipSuccess &&
              hipMalloc(&ctx->d_clv, kMaxL * sizeof(double)) == hipSuccess &&
              hipMemcpy(ctx->d_clv, clv.data(), kMaxL * sizeof(double), hipMemcpyHostToDevice) == hipSuccess &&
              hipMalloc(&ctx->d_sh, kSlotCapacity * sizeof(ShSim)) == hipSuccess &&
              hipMalloc(&ctx->d_ctl, 2 * sizeof(int)) == hipSuccess && hipMemset(ctx->d_ctl, 0, 2 * sizeof(int)) == hipSuccess &&
              hipMalloc(&ctx->d_line, kSlotCapacity * sizeof(LineSim)) == hipSuccess &&
              hipMalloc(&ctx->d_cyl, kSlotCapacity * sizeof(CylSim)) == hipSuccess &&
              hipMemset(ctx->d_sh, 0, kSlotCapacity * sizeof(ShSim)) == hipSuccess &&
              hipMemset(ctx->d_line, 0, kSlotCapacity * sizeof(LineSim)) == hipSuccess &&
              hipMemset(ctx->d_cyl, 0, kSlotCapacity * sizeof(CylSim)) == hipSuccess &&
              hipEventCreate(&ctx->ev_start) == hipSuccess && hipEventCreate(&ctx->ev_stop) == hipSuccess &&
              hipEventCreateWithFlags(&ctx->ev_fork, hipEventDisableTiming) == hipSuccess;
    for (int j = 0; ok && j < kSideStreams; ++j)
        ok = hipStreamCreateWithFlags(&ctx->side[j], hipStreamNonBlocking) == hipSuccess &&
             hipEventCreateWithFlags(&ctx->ev_join[j], hipEventDisableTiming) == hipSuccess;
    if (!ok) {
        tdse_ctx_destroy(ctx);
        return fail(nullptr, TDSE_ERR_HIP, "context allocation failed");
    }
    hipError_t se = hipSuccess;
    ctx->scratch = device_scratch(device, &se);
    if (!ctx->scratch) {
        tdse_ctx_destroy(ctx);
        return fail(nullptr, TDSE_ERR_HIP, std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(se));
    }
    *out = ctx;
    return TDSE_OK;
}

int tdse_ctx_destroy(tdse_ctx* ctx) {
    if (!ctx) return TDSE_OK;
    (void)hipSetDevice(ctx->device);
    if (ctx->stream) (void)hipStreamSynchronize(ctx->stream);
    drop_graph(ctx);
    for (auto* v : {&ctx->sh_buckets, &ctx->sh_adi_buckets, &ctx->sh_adi_lbuckets, &ctx->line_buckets,
                    &ctx->cyl_buckets})
        for (auto& b : *v) free_bucket(b);
    if (ctx->adi_waves.ptr) (void)hipFree(ctx->adi_waves.ptr);
    if (ctx->cyl_jobs.ptr) (void)hipFree(ctx->cyl_jobs.ptr);
    if (ctx->cyl_count_jobs.ptr) (void)hipFree(ctx->cyl_count_jobs.ptr);
    for (auto* v : {&ctx->adi_jobs, &ctx->any_lines, &ctx->any_pairs, &ctx->any_adi_lines, &ctx->any_adi_groups})
        if (v->ptr) (void)hipFree(v->ptr);
    if (ctx->d_cyl) (void)hipFree(ctx->d_cyl);
    if (ctx->waves.ptr) (void)hipFree(ctx->waves.ptr);
    if (ctx->jobs.ptr) (void)hipFree(ctx->jobs.ptr);
    if (ctx->d_cl) (void)hipFree(ctx->d_cl);
    if (ctx->d_clv) (void)hipFree(ctx->d_clv);
    if (ctx->d_sh) (void)hipFree(ctx->d_sh);
    if (ctx->d_ctl) (void)hipFree(ctx->d_ctl);
    if (ctx->d_line) (void)hipFree(ctx->d_line);
    for (hipEvent_t e : ctx->ev_pool) (void)hipEventDestroy(e);
    if (ctx->ev_start) (void)hipEventDestroy(ctx->ev_start);
    if (ctx->ev_stop) (void)hipEventDestroy(ctx->ev_stop);
    if (ctx->ev_fork) (void)hipEventDestroy(ctx->ev_fork);
    for (int j = 0; j < kSideStreams; ++j) {
        if (ctx->ev_join[j]) (void)hipEventDestroy(ctx->ev_join[j]);
        if (ctx->side[j]) (void)hipStreamDestroy(ctx->side[j]);
    }
    ctx->arena.release();
    if (ctx->stream) (void)hipStreamDestroy(ctx->stream);
    delete ctx;
    return TDSE_OK;
}

int tdse_sync(tdse_ctx* ctx) {
    if (!ctx) return fail(nullptr, TDSE_ERR_ARG, "ctx is NULL");
    HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
    return TDSE_OK;
}

int tdse_pool_usage(tdse_ctx* ctx, size_t* used_bytes, size_t* total_bytes) {
    if (!ctx) return fail(nullptr, TDSE_ERR_ARG, "ctx is NULL");
    if (used_bytes) *used_bytes = ctx->arena.used;
    if (total_bytes) *total_bytes = ctx->arena.size;
    return TDSE_OK;
}

int tdse_copy_probe(tdse_ctx* ctx, size_t bytes, int launches, double* avg_ms) {
    if (!ctx) return fail(nullptr, TDSE_ERR_ARG, "ctx is NULL");
    if (bytes == 0 || bytes % sizeof(double2) != 0 || launches < 1)
        return fail(ctx, TDSE_ERR_ARG, "tdse_copy_probe: bytes must be a positive multiple of 16, launches >= 1");
    HIP_TRY(ctx, hipSetDevice(ctx->device));
    std::vector<void*> blocks;
    double2 *src, *dst;
    const size_t n = bytes / sizeof(double2);
    int rc = copy_to_device<double2>(ctx, blocks, nullptr, n, &src);
    if (rc == TDSE_OK) rc = copy_to_device<double2>(ctx, blocks, nullptr, n, &dst);
    if (rc != TDSE_OK) {
        free_blocks(ctx, blocks);
        return rc;
    }
    const unsigned grid = (unsigned)std::min<size_t>((n + 255) / 256, (size_t)1 << 20);
    hipError_t e = hipEventRecord(ctx->ev_start, ctx->stream);
    for (int i = 0; i < launches && e == hipSuccess; ++i) {
        hipLaunchKernelGGL(k_stream_copy, dim3(grid), dim3(256), 0, ctx->stream, src, dst, n);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipEventRecord(ctx->ev_stop, ctx->stream);
    if (e == hipSuccess) e = hipEventSynchronize(ctx->ev_stop);
    float ms = 0.f;
    if (e == hipSuccess) e = hipEventElapsedTime(&ms, ctx->ev_start, ctx->ev_stop);
    free_blocks(ctx, blocks);
    if (e != hipSuccess) return fail(ctx, TDSE_ERR_HIP, std::string("tdse_copy_probe: ") + hipGetErrorString(e));
    if (avg_ms) *avg_ms = ms / launches;
    return TDSE_OK;
}

int tdse_tdma_batched(tdse_ctx* ctx, const double* sub, const double* diag, const double* sup, const double* d,
                      double* x, const int64_t* offsets, const int64_t* lengths, int64_t n_systems) {
    if (!ctx) return fail(nullptr, TDSE_ERR_ARG, "ctx is NULL");
    if (!sub || !diag || !sup || !d || !x || !offsets || !lengths || n_systems < 0)
        return fail(ctx, TDSE_ERR_ARG, "tdse_tdma_batched: NULL array or negative count");
    if (n_systems == 0) return TDSE_OK;
    int64_t total = 0;
    for (int64_t i = 0; i < n_systems; ++i) {
        if (lengths[i] < 1 || offsets[i] < 0) return fail(ctx, TDSE_ERR_ARG, "tdse_tdma_batched: bad system extent");
        total = std::max(total, offsets[i] + lengths[i]);
    }
    HIP_TRY(ctx, hipSetDevice(ctx->device));
    std::vector<void*> blocks;
    double2 *da, *db, *dc, *dd, *dx, *dcp;
    int64_t *doff, *dlen;
    int rc = 0;
    const size_t n = (size_t)total;
    if ((rc = copy_to_device(ctx, blocks, reinterpret_cast<const double2*>(sub), n, &da)) ||
        (rc = copy_to_device(ctx, blocks, reinterpret_cast<const double2*>(diag), n, &db)) ||
        (rc = copy_to_device(ctx, blocks, reinterpret_cast<const double2*>(sup), n, &dc)) ||
        (rc = copy_to_device(ctx, blocks, reinterpret_cast<const double2*>(d), n, &dd)) ||
        (rc = copy_to_device<double2>(ctx, blocks, nullptr, n, &dx)) ||
        (rc = copy_to_device<double2>(ctx, blocks, nullptr, n, &dcp)) ||
        (rc = copy_to_device(ctx, blocks, offsets, (size_t)n_systems, &doff)) ||
        (rc = copy_to_device(ctx, blocks, lengths, (size_t)n_systems, &dlen))) {
        (void)hipStreamSynchronize(ctx->stream);
        free_blocks(ctx, blocks);
        return rc;
    }
    hipError_t e = launch_tdma(ctx, da, db, dc, dd, dx, dcp, doff, dlen, lengths, n_systems, false);
    if (e == hipSuccess) e = hipMemcpyAsync(x, dx, n * sizeof(double2), hipMemcpyDeviceToHost, ctx->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(ctx->stream);
    (void)hipStreamSynchronize(ctx->stream);
    free_blocks(ctx, blocks);
    if (e != hipSuccess) return fail(ctx, TDSE_ERR_HIP, std::string("tdse_tdma_batched: ") + hipGetErrorString(e));
    return TDSE_OK;
}

int tdse_tdma(tdse_ctx* ctx, const double* sub, const double* diag, const double* sup, const double* d, double* x,
              int64_t n) {
    if (n < 1) return fail(ctx, TDSE_ERR_ARG, "tdse_tdma: n must be >= 1");
    const int64_t off = 0;
    return tdse_tdma_batched(ctx, sub, diag, sup, d, x, &off, &n, 1);
}

int tdse_tdma_batched_noalloc(tdse_ctx* ctx, const double* sub, const double* diag, const double* sup,
                              const double* d, double* x, const int64_t* offsets, const int64_t* lengths,
                              int64_t n_systems, int64_t total) {
    if (!ctx) return fail(nullptr, TDSE_ERR_ARG, "ctx is NULL");
    if (!sub || !diag || !sup || !d || !x || !offsets || !lengths || n_systems < 0 || total < 0)
        return fail(ctx, TDSE_ERR_ARG, "tdse_tdma_batched_noalloc: NULL array or negative count");
    if (total > kNoAllocPoints)
        return fail(ctx, TDSE_ERR_ARG, "tdse_tdma_batched_noalloc: total " + std::to_string(total) +
                                           " exceeds the scratch maximum of " + std::to_string(kNoAllocPoints) +
                                           " unknowns");
    if (n_systems > kNoAllocSystems)
        return fail(ctx, TDSE_ERR_ARG, "tdse_tdma_batched_noalloc: " + std::to_string(n_systems) +
                                           " systems exceed the scratch maximum of " +
                                           std::to_string(kNoAllocSystems));
    for (int64_t i = 0; i < n_systems; ++i)
        if (lengths[i] < 1 || offsets[i] < 0 || offsets[i] > total - lengths[i])
            return fail(ctx, TDSE_ERR_ARG, "tdse_tdma_batched_noalloc: system " + std::to_string(i) +
                                               " lies outside [0, total)");
    if (n_systems == 0) return TDSE_OK;
    if (!ctx->scratch) return fail(ctx, TDSE_ERR_STATE, "tdse_tdma_batched_noalloc: no device scratch");
    HIP_TRY(ctx, hipSetDevice(ctx->device));
    double2* cp = ctx->scratch;
    int64_t* doff = reinterpret_cast<int64_t*>(cp + kNoAllocPoints);
    int64_t* dlen = doff + kNoAllocSystems;
    const size_t nb = (size_t)n_systems * sizeof(int64_t);
    HIP_TRY(ctx, hipMemcpyAsync(doff, offsets, nb, hipMemcpyHostToDevice, ctx->stream));
    HIP_TRY(ctx, hipMemcpyAsync(dlen, lengths, nb, hipMemcpyHostToDevice, ctx->stream));
    bool in_place = false;
    for (const double* input : {sub, diag, sup, d}) in_place = in_place || (x < input + 2 * total && input < x + 2 * total);
    HIP_TRY(ctx, launch_tdma(ctx, reinterpret_cast<const double2*>(sub), reinterpret_cast<const double2*>(diag),
                             reinterpret_cast<const double2*>(sup), reinterpret_cast<const double2*>(d),
                             reinterpret_cast<double2*>(x), cp, doff, dlen, lengths, n_systems, in_place));
    HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
    return TDSE_OK;
}

int tdse_sh_add(tdse_ctx* ctx, const tdse_sh_desc* desc, const double* tables, const double* fs, const double* ts,
                const double* g0, const double* basis, const int32_t* basis_l, int32_t* slot) {
    if (!ctx) return fail(nullptr, TDSE_ERR_ARG, "ctx is NULL");
    if (!desc || !tables || !fs || !ts || !g0 || !slot) return fail(ctx, TDSE_ERR_ARG, "tdse_sh_add: NULL argument");
    const tdse_sh_desc& D = *desc;
    const int P = D.chunks, m = D.rows;
    if (D.r_points < 2 || D.l_bound < 1 || D.l_bound > kMaxL) return fail(ctx, TDSE_ERR_ARG, "tdse_sh_add: bad mesh size");
    if (P < TDSE_WAVE || P % TDSE_WAVE) return fail(ctx, TDSE_ERR_ARG, "tdse_sh_add: chunks must be a positive multiple of 64");
    if (m < 2 || m > 16 || (m & 1)) return fail(ctx, TDSE_ERR_ARG, "tdse_sh_add: rows must be even and in [2, 16]");
    if (P > 512) return fail(ctx, TDSE_ERR_ARG, "tdse_sh_add: at most 512 chunks");
    if ((int64_t)P * m < D.r_points) return fail(ctx, TDSE_ERR_ARG, "tdse_sh_add: chunks * rows < r_points");
    if (D.n_steps < 1) return fail(ctx, TDSE_ERR_ARG, "tdse_sh_add: n_steps must be >= 1");
    if (D.store_every == 0 || D.store_every < -1) return fail(ctx, TDSE_ERR_ARG, "tdse_sh_add: store_every must be >= 1 or -1");
    if (D.n_basis < 0 || (D.n_basis > 0 && (!basis || !basis_l))) return fail(ctx, TDSE_ERR_ARG, "tdse_sh_add: basis missing");
    if (D.lb < 1 || D.lb > D.l_bound) return fail(ctx, TDSE_ERR_ARG, "tdse_sh_add: lb out of range");
    if (D.gauge != 0 && D.gauge != 1) return fail(ctx, TDSE_ERR_ARG, "tdse_sh_add: gauge must be 0 (length) or 1 (velocity)");
    if (D.gauge == 1 && (D.r_points < 3 || D.l_bound < 2))
        return fail(ctx, TDSE_ERR_ARG, "tdse_sh_add: the velocity gauge needs r_points >= 3 and l_bound >= 2");
    if (D.method != 0 && D.method != 1) return fail(ctx, TDSE_ERR_ARG, "tdse_sh_add: method must be 0 or 1");
    if (D.method == 1 && D.gauge != 0)
        return fail(ctx, TDSE_ERR_ARG, "tdse_sh_add: AlternatingDirectionImplicit runs the length gauge");
    for (int b = 0; b < D.n_basis; ++b)
        if (basis_l[b] < 0 || basis_l[b] >= D.lb) return fail(ctx, TDSE_ERR_ARG, "tdse_sh_add: basis l must be < lb");
    HIP_TRY(ctx, hipSetDevice(ctx->device));
    int s = -1;
    for (int i = 0; i < (int)ctx->sh.size(); ++i)
        if (!ctx->sh[i].live) {
            s = i;
            break;
        }
    if (s < 0) {
        if ((int)ctx->sh.size() >= kSlotCapacity) return fail(ctx, TDSE_ERR_NOMEM, "no free simulation slot");
        ctx->sh.emplace_back();
        s = (int)ctx->sh.size() - 1;
    }
    ShHost& H = ctx->sh[s];
    H.blocks.clear();
    H.vel = D.gauge == 1;
    H.adi = D.method == 1;
    ShSim& S = H.dev;
    S = ShSim{};
    S.n = D.r_points;
    S.L = D.l_bound;
    S.P = P;
    S.m = m;
    S.npad = P * m;
    S.N = D.n_steps;
    S.store_every = D.store_every;
    S.LB = D.lb;
    S.n_basis = D.n_basis;
    S.n_part = (S.npad / TDSE_WAVE) * sh_parts(S.L);
    S.norm_by_l = D.norm_by_l ? 1 : 0;
    S.corr0 = D.corr0;
    S.delta_r = D.delta_r;
    S.cu = D.centrifugal;
    S.step = 0;
    S.active = 1;
    H.n_data = n_data_points(S.N, S.store_every);
    const size_t npad = S.npad;
    double2 *g, *g2, *snap, *oip, *ta;
    double *tab, *dfs, *dts, *part, *on, *oln, *bas = nullptr, *pl = nullptr, *onl = nullptr, *dfa = nullptr;
    int* bl = nullptr;
    int rc = 0;
    std::vector<double2> ta_host(npad);  // (T_j, A_j) interleaved for the R-phase
    for (size_t p = 0; p < npad; ++p) ta_host[p] = make_double2(tables[SH_IN_T * npad + p], tables[SH_IN_AN * npad + p]);
    if ((rc = copy_to_device(ctx, H.blocks, reinterpret_cast<const double2*>(g0), (size_t)S.L * npad, &g)) ||
        (rc = copy_to_device(ctx, H.blocks, ta_host.data(), npad, &ta)) ||
        (rc = copy_to_device<double2>(ctx, H.blocks, nullptr, (size_t)S.L * npad, &g2)) ||
        (rc = copy_to_device(ctx, H.blocks, tables + SH_IN_AN * npad, (SH_NTAB - SH_IN_AN + (H.vel ? 1 : 0)) * npad, &tab)) ||
        // ADI: the L-phase sees a zero field (it only masks and observes); the field goes to fa
        (rc = copy_to_device(ctx, H.blocks, H.adi ? nullptr : fs, (size_t)S.N, &dfs)) ||
        (H.adi && (rc = copy_to_device(ctx, H.blocks, fs, (size_t)S.N, &dfa))) ||
        (rc = copy_to_device(ctx, H.blocks, ts, (size_t)S.N, &dts)) ||
        (rc = copy_to_device<double2>(ctx, H.blocks, nullptr, (size_t)S.LB * npad, &snap)) ||
        (rc = copy_to_device<double>(ctx, H.blocks, nullptr, (size_t)S.n_part + S.npad / TDSE_WAVE, &part)) ||
        (rc = copy_to_device<double>(ctx, H.blocks, nullptr, (size_t)H.n_data, &on)) ||
        (rc = copy_to_device<double>(ctx, H.blocks, nullptr, (size_t)H.n_data, &oln)) ||
        (rc = copy_to_device<double2>(ctx, H.blocks, nullptr, (size_t)H.n_data * std::max(1, S.n_basis), &oip)) ||
        (S.n_basis > 0 && ((rc = copy_to_device(ctx, H.blocks, basis, (size_t)S.n_basis * npad, &bas)) ||
                           (rc = copy_to_device(ctx, H.blocks, basis_l, (size_t)S.n_basis, &bl)))) ||
        (S.norm_by_l &&
         ((rc = copy_to_device<double>(ctx, H.blocks, nullptr, (size_t)S.L * (S.npad / TDSE_WAVE), &pl)) ||
          (rc = copy_to_device<double>(ctx, H.blocks, nullptr, (size_t)H.n_data * S.L, &onl))))) {
        (void)hipStreamSynchronize(ctx->stream);
        free_blocks(ctx, H.blocks);
        return rc;
    }
    S.g = g;
    S.g2 = g2;
    S.ta = ta;
    S.tab = tab;
    S.fs = dfs;
    S.ts = dts;
    S.snap = snap;
    S.part = part;
    S.out_norm = on;
    S.out_lnorm = oln;
    S.out_ip = oip;
    S.basis = bas;
    S.basis_l = bl;
    S.part_l = pl;
    S.out_nl = onl;
    S.fa = dfa;
    S.adi = H.adi ? 1 : 0;
    HIP_TRY(ctx, hipMemcpyAsync(ctx->d_sh + s, &S, sizeof(ShSim), hipMemcpyHostToDevice, ctx->stream));
    HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));  // host buffers may be released after return
    H.live = true;
    ctx->dirty = true;
    *slot = s;
    return TDSE_OK;
}

int tdse_line_add(tdse_ctx* ctx, const tdse_line_desc* desc, const double* tables, const double* wt, const double* fs,
                  const double* g0, const double* basis, int32_t* slot) {
    if (!ctx) return fail(nullptr, TDSE_ERR_ARG, "ctx is NULL");
    if (!desc || !tables || !wt || !fs || !g0 || !slot) return fail(ctx, TDSE_ERR_ARG, "tdse_line_add: NULL argument");
    const tdse_line_desc& D = *desc;
    const int P = D.chunks, m = D.rows;
    if (D.z_points < 2) return fail(ctx, TDSE_ERR_ARG, "tdse_line_add: z_points must be >= 2");
    if (P < TDSE_WAVE || P % TDSE_WAVE) return fail(ctx, TDSE_ERR_ARG, "tdse_line_add: chunks must be a positive multiple of 64");
    if (m < 2 || m > 16 || (m & 1)) return fail(ctx, TDSE_ERR_ARG, "tdse_line_add: rows must be even and in [2, 16]");
    if (P > 512) return fail(ctx, TDSE_ERR_ARG, "tdse_line_add: chunks must be <= 512");
    if ((int64_t)P * m < D.z_points) return fail(ctx, TDSE_ERR_ARG, "tdse_line_add: chunks * rows < z_points");
    if (D.n_steps < 1) return fail(ctx, TDSE_ERR_ARG, "tdse_line_add: n_steps must be >= 1");
    if (D.store_every == 0 || D.store_every < -1) return fail(ctx, TDSE_ERR_ARG, "tdse_line_add: store_every must be >= 1 or -1");
    if (D.n_basis < 0 || (D.n_basis > 0 && !basis)) return fail(ctx, TDSE_ERR_ARG, "tdse_line_add: basis missing");
    if (D.method < 0 || D.method > 2) return fail(ctx, TDSE_ERR_ARG, "tdse_line_add: method must be 0, 1 or 2");
    if (D.method != 0 && D.renormalize)
        return fail(ctx, TDSE_ERR_ARG, "tdse_line_add: the split operator does not renormalise");
    HIP_TRY(ctx, hipSetDevice(ctx->device));
    int s = -1;
    for (int i = 0; i < (int)ctx->line.size(); ++i)
        if (!ctx->line[i].live) {
            s = i;
            break;
        }
    if (s < 0) {
        if ((int)ctx->line.size() >= kSlotCapacity) return fail(ctx, TDSE_ERR_NOMEM, "no free simulation slot");
        ctx->line.emplace_back();
        s = (int)ctx->line.size() - 1;
    }
    LineHost& H = ctx->line[s];
    H.blocks.clear();
    H.complex_steps = false;
    for (int i = 0; i < D.n_steps; ++i)
        if (wt[2 * i] != 0.0) H.complex_steps = true;
    if (D.method != 0 && H.complex_steps)
        return fail(ctx, TDSE_ERR_ARG, "tdse_line_add: the split operator needs real time steps");
    LineSim& S = H.dev;
    S = LineSim{};
    S.n = D.z_points;
    S.P = P;
    S.m = m;
    S.npad = P * m;
    S.N = D.n_steps;
    S.store_every = D.store_every;
    S.n_basis = D.n_basis;
    S.renormalize = D.renormalize;
    S.delta_z = D.delta_z;
    S.off = D.offdiag;
    S.zq0 = D.zq_first;
    S.dzq = D.zq_step;
    S.vq = D.vel_factor;
    S.method = D.method;
    S.step = 0;
    S.active = 1;
    H.n_data = n_data_points(S.N, S.store_every);
    const size_t npad = S.npad;
    double2 *g, *dwt, *oip, *bas = nullptr;
    double *tab, *dfs, *on;
    int rc = 0;
    if ((rc = copy_to_device(ctx, H.blocks, reinterpret_cast<const double2*>(g0), npad, &g)) ||
        (rc = copy_to_device(ctx, H.blocks, tables, LN_NTAB * npad, &tab)) ||
        (rc = copy_to_device(ctx, H.blocks, reinterpret_cast<const double2*>(wt), (size_t)S.N, &dwt)) ||
        (rc = copy_to_device(ctx, H.blocks, fs, (size_t)S.N, &dfs)) ||
        (rc = copy_to_device<double>(ctx, H.blocks, nullptr, (size_t)H.n_data, &on)) ||
        (rc = copy_to_device<double2>(ctx, H.blocks, nullptr, (size_t)H.n_data * std::max(1, S.n_basis), &oip)) ||
        (S.n_basis > 0 &&
         (rc = copy_to_device(ctx, H.blocks, reinterpret_cast<const double2*>(basis), (size_t)S.n_basis * npad, &bas)))) {
        (void)hipStreamSynchronize(ctx->stream);
        free_blocks(ctx, H.blocks);
        return rc;
    }
    S.g = g;
    S.tab = tab;
    S.wt = dwt;
    S.fs = dfs;
    S.out_norm = on;
    S.out_ip = oip;
    S.basis = bas;
    HIP_TRY(ctx, hipMemcpyAsync(ctx->d_line + s, &S, sizeof(LineSim), hipMemcpyHostToDevice, ctx->stream));
    HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));  // host buffers may be released after return
    H.live = true;
    ctx->dirty = true;
    *slot = s;
    return TDSE_OK;
}

int tdse_cyl_add(tdse_ctx* ctx, const tdse_cyl_desc* desc, const double* zt, const double* rt, const double* roff,
                 const double* fs, const double* ts, const double* g0, const double* basis, int32_t* slot) {
    if (!ctx) return fail(nullptr, TDSE_ERR_ARG, "ctx is NULL");
    if (!desc || !zt || !rt || !roff || !fs || !ts || !g0 || !slot)
        return fail(ctx, TDSE_ERR_ARG, "tdse_cyl_add: NULL argument");
    const tdse_cyl_desc& D = *desc;
    if (D.z_points < 2 || D.rho_points < 2) return fail(ctx, TDSE_ERR_ARG, "tdse_cyl_add: bad mesh size");
    const int Pz = D.z_chunks, Mz = D.z_rows, Cr = D.rho_chunks, Mr = D.rho_rows, lanes = D.lanes;
    if (Pz < TDSE_WAVE || Pz % TDSE_WAVE) return fail(ctx, TDSE_ERR_ARG, "tdse_cyl_add: z_chunks must be a positive multiple of 64");
    if (Mz < 2 || Mz > 16 || (Mz & 1)) return fail(ctx, TDSE_ERR_ARG, "tdse_cyl_add: z_rows must be even and in [2, 16]");
    if ((Mz <= 8 && Pz > 512) || (Mz > 8 && Pz > 256)) return fail(ctx, TDSE_ERR_ARG, "tdse_cyl_add: too many z chunks for z rows");
    if ((int64_t)Pz * Mz < D.z_points) return fail(ctx, TDSE_ERR_ARG, "tdse_cyl_add: z_chunks * z_rows < z_points");
    const bool shape_ok = (Mr == 4 && lanes == 4 && Cr * 4 <= 1024) || (Mr == 8 && lanes == 4 && Cr * 4 <= 512) ||
                          (Mr == 4 && lanes == 8 && Cr * 8 <= 1024) || (Mr == 8 && lanes == 8 && Cr * 8 <= 1024) ||
                          (Mr == 16 && lanes == 4 && Cr * 4 <= 512);
    if (!shape_ok || Cr < 1 || (Cr * lanes) % TDSE_WAVE)
        return fail(ctx, TDSE_ERR_ARG, "tdse_cyl_add: unsupported rho layout (rows, lanes, chunks)");
    if ((int64_t)Cr * Mr < D.rho_points) return fail(ctx, TDSE_ERR_ARG, "tdse_cyl_add: rho_chunks * rho_rows < rho_points");
    if (D.n_steps < 1) return fail(ctx, TDSE_ERR_ARG, "tdse_cyl_add: n_steps must be >= 1");
    if (D.store_every == 0 || D.store_every < -1) return fail(ctx, TDSE_ERR_ARG, "tdse_cyl_add: store_every must be >= 1 or -1");
    if (D.n_basis < 0 || (D.n_basis > 0 && !basis)) return fail(ctx, TDSE_ERR_ARG, "tdse_cyl_add: basis missing");
    HIP_TRY(ctx, hipSetDevice(ctx->device));
    int s = -1;
    for (int i = 0; i < (int)ctx->cyl.size(); ++i)
        if (!ctx->cyl[i].live) {
            s = i;
            break;
        }
    if (s < 0) {
        if ((int)ctx->cyl.size() >= kSlotCapacity) return fail(ctx, TDSE_ERR_NOMEM, "no free simulation slot");
        ctx->cyl.emplace_back();
        s = (int)ctx->cyl.size() - 1;
    }
    CylHost& H = ctx->cyl[s];
    H.blocks.clear();
    CylSim& S = H.dev;
    S = CylSim{};
    S.nz = D.z_points;
    S.nr = D.rho_points;
    S.Pz = Pz;
    S.Mz = Mz;
    S.npz = Pz * Mz;
    S.Cr = Cr;
    S.Mr = Mr;
    S.nrpad = Cr * Mr;
    S.lanes = lanes;
    S.n_groups = S.npz / lanes;
    S.N = D.n_steps;
    S.store_every = D.store_every;
    S.n_basis = D.n_basis;
    S.zp = D.z_prefactor;
    S.rp = D.rho_prefactor;
    S.kc = D.coulomb;
    S.q = D.test_charge;
    S.delta = D.delta;
    S.has_mask = D.has_mask;
    S.m_inner = D.mask_inner;
    S.m_outer = D.mask_outer;
    S.m_inv_s = D.mask_smoothness > 0 ? 1.0 / D.mask_smoothness : 1.0;
    S.m_roots = -1;
    for (int k = 0; k <= 10; ++k)
        if (D.mask_smoothness == (double)(1 << k)) S.m_roots = k;
    S.z0 = D.z_first;
    S.dz = D.z_step;
    S.rho0 = D.rho_first;
    S.drho = D.rho_step;
    S.step = 0;
    S.obs = -1;
    S.active = 1;
    S.phase = 1;
    S.hold = 0;
    H.n_data = n_data_points(S.N, S.store_every);
    const size_t pts = (size_t)S.nrpad * S.npz;
    double2 *g, *oip, *bas = nullptr;
    double *dzt, *droff, *dfs, *dts, *part, *on;
    // rp c(j + 1) in the rho-sweep's order, from the descriptor (not rt and roff); rounded three times. The same at every
    // step, a rounding adds up as a phase: after 1000 steps of 250 x 100 the wavefunction is 2.4e-13 from one in long
    // double with the same prefactors (2.4e-13 too with one rounding; 6.1e-13 when the kernels formed the couplings).
    std::vector<double> coupling((size_t)S.nrpad, 0.0);
    for (int j = 0; j + 1 < S.nr; ++j) {
        const double m = j + 1;
        coupling[(size_t)(j % Mr) * Cr + j / Mr] = (m * (1.0 / std::sqrt(m * m - 0.25))) * S.rp;
    }
    int rc = 0;
    if ((rc = copy_to_device(ctx, H.blocks, reinterpret_cast<const double2*>(g0), pts, &g)) ||
        (rc = copy_to_device(ctx, H.blocks, zt, (size_t)S.npz, &dzt)) ||
        (rc = copy_to_device(ctx, H.blocks, coupling.data(), coupling.size(), &droff)) ||
        (rc = copy_to_device(ctx, H.blocks, fs, (size_t)S.N, &dfs)) ||
        (rc = copy_to_device(ctx, H.blocks, ts, (size_t)S.N, &dts)) ||
        (rc = copy_to_device<double>(ctx, H.blocks, nullptr, (size_t)S.n_groups * (1 + 2 * S.n_basis), &part)) ||
        (rc = copy_to_device<double>(ctx, H.blocks, nullptr, (size_t)H.n_data, &on)) ||
        (rc = copy_to_device<double2>(ctx, H.blocks, nullptr, (size_t)H.n_data * std::max(1, S.n_basis), &oip)) ||
        (S.n_basis > 0 &&
         (rc = copy_to_device(ctx, H.blocks, reinterpret_cast<const double2*>(basis), (size_t)S.n_basis * pts, &bas)))) {
        (void)hipStreamSynchronize(ctx->stream);
        free_blocks(ctx, H.blocks);
        return rc;
    }
    S.g = g;
    S.zt = dzt;
    S.roff = droff;
    S.fs = dfs;
    S.ts = dts;
    S.part = part;
    S.out_norm = on;
    S.out_ip = oip;
    S.basis = bas;
    HIP_TRY(ctx, hipMemcpyAsync(ctx->d_cyl + s, &S, sizeof(CylSim), hipMemcpyHostToDevice, ctx->stream));
    HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));  // host buffers may be released after return
    H.live = true;
    ctx->dirty = true;
    ctx->cyl_pending = true;
    *slot = s;
    return TDSE_OK;
}

int tdse_set_hold(tdse_ctx* ctx, int32_t kind, int32_t slot, int32_t hold) {
    if (!ctx) return fail(nullptr, TDSE_ERR_ARG, "ctx is NULL");
    if (kind == 0 || kind == 1) return TDSE_OK;  // SH and Line states can be made exact at any step
    if (kind != 2) return fail(ctx, TDSE_ERR_ARG, "unknown simulation kind");
    if (slot < 0 || slot >= (int)ctx->cyl.size() || !ctx->cyl[slot].live) return fail(ctx, TDSE_ERR_ARG, "bad Cyl slot");
    HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
    const int h = hold ? 1 : 0;
    ctx->cyl[slot].dev.hold = h;
    HIP_TRY(ctx, hipMemcpy(reinterpret_cast<char*>(ctx->d_cyl + slot) + offsetof(CylSim, hold), &h, sizeof(int),
                           hipMemcpyHostToDevice));
    return TDSE_OK;
}

int tdse_run(tdse_ctx* ctx, int32_t n_steps, int32_t use_graph) {
    if (!ctx) return fail(nullptr, TDSE_ERR_ARG, "ctx is NULL");
    if (n_steps < 0) return fail(ctx, TDSE_ERR_ARG, "tdse_run: n_steps must be >= 0");
    HIP_TRY(ctx, hipSetDevice(ctx->device));
    int rc;
    if (ctx->dirty && (rc = rebuild_tables(ctx))) return rc;
    const bool graph = use_graph && !ctx->profiling;
    bool hold_any = false;
    for (const auto& h : ctx->cyl)
        if (h.live && h.dev.hold) hold_any = true;
    ctx->ev_used = 0;
    ctx->ev_pairs.clear();
    // SH ADI simulations may run ahead into the next step on every replay of this run but
    // the last, so that the run ends with every simulation at an ordinary step boundary
    // (mask pending) which the host can materialise, download or checkpoint.
    const bool ahead = !ctx->sh_adi_buckets.empty() && n_steps > 1;
    HIP_TRY(ctx, hipEventRecord(ctx->ev_start, ctx->stream));
    if (!ctx->sh_adi_buckets.empty())
        HIP_TRY(ctx, hipMemsetD32Async(reinterpret_cast<hipDeviceptr_t>(ctx->d_ctl), ahead ? 1 : 0, 1, ctx->stream));
    for (int i = 0; i < n_steps;) {
        // the pre-sweep is needed for simulations held at exact states, and for
        // one step after a cylindrical simulation was added or uploaded
        int done = 1;
        const int left = n_steps - i - (ahead ? 1 : 0);  // steps before the last one of a run with run-ahead
        if (ahead && left == 0)
            HIP_TRY(ctx, hipMemsetD32Async(reinterpret_cast<hipDeviceptr_t>(ctx->d_ctl), 0, 1, ctx->stream));
        if (ctx->cyl_pending && !hold_any) {
            if ((rc = launch_step(ctx, true))) return rc;
        } else if (graph) {
            if ((rc = ensure_graph(ctx, hold_any))) return rc;
            if (kGraphSteps > 1 && left >= kGraphSteps) {
                HIP_TRY(ctx, hipGraphLaunch(ctx->exec_k, ctx->stream));
                done = kGraphSteps;
            } else {
                HIP_TRY(ctx, hipGraphLaunch(ctx->exec, ctx->stream));
            }
        } else if ((rc = launch_step(ctx, hold_any))) {
            return rc;
        }
        ctx->cyl_pending = false;
        i += done;
    }
    if (n_steps > 0 && !ctx->cyl_buckets.empty()) {  // the last step's observations
        cyl_observe(ctx);
        HIP_TRY(ctx, hipGetLastError());
    }
    HIP_TRY(ctx, hipEventRecord(ctx->ev_stop, ctx->stream));
    HIP_TRY(ctx, hipEventSynchronize(ctx->ev_stop));
    float ms = 0.f;
    HIP_TRY(ctx, hipEventElapsedTime(&ms, ctx->ev_start, ctx->ev_stop));
    ctx->last_run_ms = ms;
    if (ctx->profiling) {
        for (auto& pr : ctx->ev_pairs) {
            float t = 0.f;
            HIP_TRY(ctx, hipEventElapsedTime(&t, ctx->ev_pool[pr.second], ctx->ev_pool[pr.second + 1]));
            ctx->prof_ms[pr.first] += t;
            ctx->prof_n[pr.first] += 1;
        }
    }
    return TDSE_OK;
}

int tdse_line_run(tdse_ctx* ctx, int32_t n_steps) {
    if (!ctx) return fail(nullptr, TDSE_ERR_ARG, "ctx is NULL");
    if (n_steps < 0) return fail(ctx, TDSE_ERR_ARG, "tdse_line_run: n_steps must be >= 0");
    HIP_TRY(ctx, hipSetDevice(ctx->device));
    int rc;
    if (ctx->dirty && (rc = rebuild_tables(ctx))) return rc;
    HIP_TRY(ctx, hipEventRecord(ctx->ev_start, ctx->stream));
    if ((rc = fan_out(ctx, ctx->line_buckets,
                      [&](const Bucket& b, hipStream_t st) { dispatch_line(ctx, b, n_steps, st); })))
        return rc;
    HIP_TRY(ctx, hipGetLastError());
    HIP_TRY(ctx, hipEventRecord(ctx->ev_stop, ctx->stream));
    HIP_TRY(ctx, hipEventSynchronize(ctx->ev_stop));
    float ms = 0.f;
    HIP_TRY(ctx, hipEventElapsedTime(&ms, ctx->ev_start, ctx->ev_stop));
    ctx->last_run_ms = ms;
    return TDSE_OK;
}

int tdse_sim_state(tdse_ctx* ctx, int32_t kind, int32_t slot, int32_t* step, int32_t* n_steps, int32_t* n_data) {
    if (!ctx) return fail(nullptr, TDSE_ERR_ARG, "ctx is NULL");
    HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
    int st = 0;
    if (kind == 0) {
        if (slot < 0 || slot >= (int)ctx->sh.size() || !ctx->sh[slot].live) return fail(ctx, TDSE_ERR_ARG, "bad SH slot");
        HIP_TRY(ctx, hipMemcpy(&st, reinterpret_cast<char*>(ctx->d_sh + slot) + offsetof(ShSim, step), sizeof(int),
                               hipMemcpyDeviceToHost));
        if (n_steps) *n_steps = ctx->sh[slot].dev.N;
        if (n_data) *n_data = ctx->sh[slot].n_data;
    } else if (kind == 1) {
        if (slot < 0 || slot >= (int)ctx->line.size() || !ctx->line[slot].live)
            return fail(ctx, TDSE_ERR_ARG, "bad Line slot");
        HIP_TRY(ctx, hipMemcpy(&st, reinterpret_cast<char*>(ctx->d_line + slot) + offsetof(LineSim, step), sizeof(int),
                               hipMemcpyDeviceToHost));
        if (n_steps) *n_steps = ctx->line[slot].dev.N;
        if (n_data) *n_data = ctx->line[slot].n_data;
    } else if (kind == 2) {
        if (slot < 0 || slot >= (int)ctx->cyl.size() || !ctx->cyl[slot].live) return fail(ctx, TDSE_ERR_ARG, "bad Cyl slot");
        HIP_TRY(ctx, hipMemcpy(&st, reinterpret_cast<char*>(ctx->d_cyl + slot) + offsetof(CylSim, step), sizeof(int),
                               hipMemcpyDeviceToHost));
        if (n_steps) *n_steps = ctx->cyl[slot].dev.N;
        if (n_data) *n_data = ctx->cyl[slot].n_data;
    } else {
        return fail(ctx, TDSE_ERR_ARG, "unknown simulation kind");
    }
    if (step) *step = st;
    return TDSE_OK;
}

int tdse_download(tdse_ctx* ctx, int32_t kind, int32_t slot, double* g, double* norms, double* lnorms, double* ips) {
    if (!ctx) return fail(nullptr, TDSE_ERR_ARG, "ctx is NULL");
    HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
    if (kind == 0) {
        if (slot < 0 || slot >= (int)ctx->sh.size() || !ctx->sh[slot].live) return fail(ctx, TDSE_ERR_ARG, "bad SH slot");
        const ShHost& H = ctx->sh[slot];
        const ShSim& S = H.dev;
        if (g) {
            int st = 0;
            HIP_TRY(ctx, hipMemcpy(&st, reinterpret_cast<char*>(ctx->d_sh + slot) + offsetof(ShSim, step), sizeof(int),
                                   hipMemcpyDeviceToHost));
            HIP_TRY(ctx, hipMemcpy(g, sh_state(S, st), (size_t)S.L * S.npad * sizeof(double2), hipMemcpyDeviceToHost));
        }
        if (norms) HIP_TRY(ctx, hipMemcpy(norms, S.out_norm, H.n_data * sizeof(double), hipMemcpyDeviceToHost));
        if (lnorms) HIP_TRY(ctx, hipMemcpy(lnorms, S.out_lnorm, H.n_data * sizeof(double), hipMemcpyDeviceToHost));
        if (ips && S.n_basis > 0)
            HIP_TRY(ctx, hipMemcpy(ips, S.out_ip, (size_t)H.n_data * S.n_basis * sizeof(double2), hipMemcpyDeviceToHost));
    } else if (kind == 1) {
        if (slot < 0 || slot >= (int)ctx->line.size() || !ctx->line[slot].live)
            return fail(ctx, TDSE_ERR_ARG, "bad Line slot");
        const LineHost& H = ctx->line[slot];
        const LineSim& S = H.dev;
        if (g) HIP_TRY(ctx, hipMemcpy(g, S.g, (size_t)S.npad * sizeof(double2), hipMemcpyDeviceToHost));
        if (norms) HIP_TRY(ctx, hipMemcpy(norms, S.out_norm, H.n_data * sizeof(double), hipMemcpyDeviceToHost));
        if (ips && S.n_basis > 0)
            HIP_TRY(ctx, hipMemcpy(ips, S.out_ip, (size_t)H.n_data * S.n_basis * sizeof(double2), hipMemcpyDeviceToHost));
    } else if (kind == 2) {
        if (slot < 0 || slot >= (int)ctx->cyl.size() || !ctx->cyl[slot].live) return fail(ctx, TDSE_ERR_ARG, "bad Cyl slot");
        const CylHost& H = ctx->cyl[slot];
        const CylSim& S = H.dev;
        if (g) HIP_TRY(ctx, hipMemcpy(g, S.g, (size_t)S.nrpad * S.npz * sizeof(double2), hipMemcpyDeviceToHost));
        if (norms) HIP_TRY(ctx, hipMemcpy(norms, S.out_norm, H.n_data * sizeof(double), hipMemcpyDeviceToHost));
        if (ips && S.n_basis > 0)
            HIP_TRY(ctx, hipMemcpy(ips, S.out_ip, (size_t)H.n_data * S.n_basis * sizeof(double2), hipMemcpyDeviceToHost));
    } else {
        return fail(ctx, TDSE_ERR_ARG, "unknown simulation kind");
    }
    return TDSE_OK;
}

int tdse_download_g(tdse_ctx* ctx, int32_t kind, int32_t slot, double* g) {
    if (!ctx) return fail(nullptr, TDSE_ERR_ARG, "ctx is NULL");
    if (!g) return fail(ctx, TDSE_ERR_ARG, "g is NULL");
    NaturalMap map;
    if (!natural_of(ctx, kind, slot, &map)) return fail(ctx, TDSE_ERR_ARG, "bad simulation kind or slot");
    HIP_TRY(ctx, hipSetDevice(ctx->device));
    HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
    double2* dev = kind == 1 ? ctx->line[slot].dev.g : kind == 2 ? ctx->cyl[slot].dev.g : nullptr;
    if (kind == 0) {
        int st = 0;
        HIP_TRY(ctx, hipMemcpy(&st, reinterpret_cast<char*>(ctx->d_sh + slot) + offsetof(ShSim, step), sizeof(int),
                               hipMemcpyDeviceToHost));
        dev = sh_state(ctx->sh[slot].dev, st);
    }
    return move_natural<true>(ctx, dev, map, reinterpret_cast<double2*>(g));
}

int tdse_download_norm_by_l(tdse_ctx* ctx, int32_t slot, double* out) {
    if (!ctx) return fail(nullptr, TDSE_ERR_ARG, "ctx is NULL");
    if (!out) return fail(ctx, TDSE_ERR_ARG, "out is NULL");
    if (slot < 0 || slot >= (int)ctx->sh.size() || !ctx->sh[slot].live) return fail(ctx, TDSE_ERR_ARG, "bad SH slot");
    const ShHost& H = ctx->sh[slot];
    if (!H.dev.norm_by_l) return fail(ctx, TDSE_ERR_STATE, "simulation was added without norm_by_l");
    HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
    HIP_TRY(ctx, hipMemcpy(out, H.dev.out_nl, (size_t)H.n_data * H.dev.L * sizeof(double), hipMemcpyDeviceToHost));
    return TDSE_OK;
}

// natural: g is in the reference's order, else in position order
static int upload_state(tdse_ctx* ctx, int32_t kind, int32_t slot, const double* g, int32_t step, bool natural) {
    if (!ctx) return fail(nullptr, TDSE_ERR_ARG, "ctx is NULL");
    if (!g) return fail(ctx, TDSE_ERR_ARG, "g is NULL");
    HIP_TRY(ctx, hipSetDevice(ctx->device));
    HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
    // other: the SH mesh's second buffer, whose padding the sweeps read and write as they do dev's
    auto copy = [&](double2* dev, size_t count, double2* other = nullptr) -> int {
        NaturalMap map;
        if (!natural_of(ctx, kind, slot, &map)) return fail(ctx, TDSE_ERR_ARG, "bad simulation kind or slot");
        if (natural)
            return move_natural<false>(ctx, dev, map, const_cast<double2*>(reinterpret_cast<const double2*>(g)),
                                       PaddedStates{dev, other});
        HIP_TRY(ctx, hipMemcpy(dev, g, count * sizeof(double2), hipMemcpyHostToDevice));
        if (other && map.padding()) {
            hipLaunchKernelGGL(k_natural<false>, dim3((unsigned)((map.padding() + 255) / 256)), dim3(256), 0, ctx->stream,
                               dev, dev, map, int64_t(0), int64_t(0), PaddedStates{other, nullptr});
            HIP_TRY(ctx, hipGetLastError());
        }
        return TDSE_OK;
    };
    int rc;
    if (kind == 0) {
        if (slot < 0 || slot >= (int)ctx->sh.size() || !ctx->sh[slot].live) return fail(ctx, TDSE_ERR_ARG, "bad SH slot");
        const ShSim& S = ctx->sh[slot].dev;
        if (step < 0 || step > S.N + 1) return fail(ctx, TDSE_ERR_ARG, "step out of range");
        if ((rc = copy(sh_state(S, step), (size_t)S.L * S.npad, sh_state(S, step + 1)))) return rc;
        const int st[2] = {step, 1};  // the uploaded g is the reference g after `step` steps
        HIP_TRY(ctx, hipMemcpy(reinterpret_cast<char*>(ctx->d_sh + slot) + offsetof(ShSim, step), &st[0], sizeof(int),
                               hipMemcpyHostToDevice));
        HIP_TRY(ctx, hipMemcpy(reinterpret_cast<char*>(ctx->d_sh + slot) + offsetof(ShSim, phase), &st[1], sizeof(int),
                               hipMemcpyHostToDevice));
        HIP_TRY(ctx, hipMemcpy(reinterpret_cast<char*>(ctx->d_sh + slot) + offsetof(ShSim, flags), &kNoFlags,
                               sizeof(int), hipMemcpyHostToDevice));
    } else if (kind == 1) {
        if (slot < 0 || slot >= (int)ctx->line.size() || !ctx->line[slot].live)
            return fail(ctx, TDSE_ERR_ARG, "bad Line slot");
        const LineSim& S = ctx->line[slot].dev;
        if (step < 0 || step > S.N + 1) return fail(ctx, TDSE_ERR_ARG, "step out of range");
        if ((rc = copy(S.g, (size_t)S.npad))) return rc;
        HIP_TRY(ctx, hipMemcpy(reinterpret_cast<char*>(ctx->d_line + slot) + offsetof(LineSim, step), &step, sizeof(int),
                               hipMemcpyHostToDevice));
        HIP_TRY(ctx, hipMemcpy(reinterpret_cast<char*>(ctx->d_line + slot) + offsetof(LineSim, flags), &kNoFlags,
                               sizeof(int), hipMemcpyHostToDevice));
    } else if (kind == 2) {
        if (slot < 0 || slot >= (int)ctx->cyl.size() || !ctx->cyl[slot].live) return fail(ctx, TDSE_ERR_ARG, "bad Cyl slot");
        const CylSim& S = ctx->cyl[slot].dev;
        if (step < 0 || step > S.N) return fail(ctx, TDSE_ERR_ARG, "step out of range");
        if ((rc = copy(S.g, (size_t)S.nrpad * S.npz))) return rc;
        const int st[2] = {step, 1};  // the uploaded g is the reference g after `step` steps
        char* base = reinterpret_cast<char*>(ctx->d_cyl + slot);
        HIP_TRY(ctx, hipMemcpy(base + offsetof(CylSim, step), &st[0], sizeof(int), hipMemcpyHostToDevice));
        HIP_TRY(ctx, hipMemcpy(base + offsetof(CylSim, phase), &st[1], sizeof(int), hipMemcpyHostToDevice));
        HIP_TRY(ctx, hipMemcpy(base + offsetof(CylSim, flags), &kNoFlags, sizeof(int), hipMemcpyHostToDevice));
        HIP_TRY(ctx, hipMemcpy(base + offsetof(CylSim, obs), &kNoObs, sizeof(int), hipMemcpyHostToDevice));
        ctx->cyl_pending = true;
    } else {
        return fail(ctx, TDSE_ERR_ARG, "unknown simulation kind");
    }
    return TDSE_OK;
}

int tdse_upload_state(tdse_ctx* ctx, int32_t kind, int32_t slot, const double* g, int32_t step) {
    return upload_state(ctx, kind, slot, g, step, false);
}

int tdse_upload_g(tdse_ctx* ctx, int32_t kind, int32_t slot, const double* g, int32_t step) {
    return upload_state(ctx, kind, slot, g, step, true);
}

int tdse_remove(tdse_ctx* ctx, int32_t kind, int32_t slot) {
    if (!ctx) return fail(nullptr, TDSE_ERR_ARG, "ctx is NULL");
    HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
    const int zero = 0;
    if (kind == 0) {
        if (slot < 0 || slot >= (int)ctx->sh.size() || !ctx->sh[slot].live) return fail(ctx, TDSE_ERR_ARG, "bad SH slot");
        HIP_TRY(ctx, hipMemcpy(reinterpret_cast<char*>(ctx->d_sh + slot) + offsetof(ShSim, active), &zero, sizeof(int),
                               hipMemcpyHostToDevice));
        free_blocks(ctx, ctx->sh[slot].blocks);
        ctx->sh[slot].live = false;
    } else if (kind == 1) {
        if (slot < 0 || slot >= (int)ctx->line.size() || !ctx->line[slot].live)
            return fail(ctx, TDSE_ERR_ARG, "bad Line slot");
        HIP_TRY(ctx, hipMemcpy(reinterpret_cast<char*>(ctx->d_line + slot) + offsetof(LineSim, active), &zero,
                               sizeof(int), hipMemcpyHostToDevice));
        free_blocks(ctx, ctx->line[slot].blocks);
        ctx->line[slot].live = false;
    } else if (kind == 2) {
        if (slot < 0 || slot >= (int)ctx->cyl.size() || !ctx->cyl[slot].live) return fail(ctx, TDSE_ERR_ARG, "bad Cyl slot");
        HIP_TRY(ctx, hipMemcpy(reinterpret_cast<char*>(ctx->d_cyl + slot) + offsetof(CylSim, active), &zero, sizeof(int),
                               hipMemcpyHostToDevice));
        free_blocks(ctx, ctx->cyl[slot].blocks);
        ctx->cyl[slot].live = false;
    } else {
        return fail(ctx, TDSE_ERR_ARG, "unknown simulation kind");
    }
    ctx->dirty = true;
    return TDSE_OK;
}

int tdse_sim_flags(tdse_ctx* ctx, int32_t kind, int32_t first_slot, int32_t n_slots, int32_t* flags) {
    if (!ctx) return fail(nullptr, TDSE_ERR_ARG, "ctx is NULL");
    if (!flags || first_slot < 0 || n_slots < 0) return fail(ctx, TDSE_ERR_ARG, "tdse_sim_flags: bad arguments");
    size_t count, pitch, off;
    const char* base;
    if (kind == 0) {
        count = ctx->sh.size(), pitch = sizeof(ShSim), off = offsetof(ShSim, flags);
        base = reinterpret_cast<const char*>(ctx->d_sh);
    } else if (kind == 1) {
        count = ctx->line.size(), pitch = sizeof(LineSim), off = offsetof(LineSim, flags);
        base = reinterpret_cast<const char*>(ctx->d_line);
    } else if (kind == 2) {
        count = ctx->cyl.size(), pitch = sizeof(CylSim), off = offsetof(CylSim, flags);
        base = reinterpret_cast<const char*>(ctx->d_cyl);
    } else {
        return fail(ctx, TDSE_ERR_ARG, "unknown simulation kind");
    }
    if ((size_t)first_slot + (size_t)n_slots > count) return fail(ctx, TDSE_ERR_ARG, "tdse_sim_flags: slot range");
    if (n_slots == 0) return TDSE_OK;
    HIP_TRY(ctx, hipSetDevice(ctx->device));
    HIP_TRY(ctx, hipMemcpy2DAsync(flags, sizeof(int32_t), base + (size_t)first_slot * pitch + off, pitch,
                                  sizeof(int32_t), (size_t)n_slots, hipMemcpyDeviceToHost, ctx->stream));
    HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
    return TDSE_OK;
}

int tdse_materialize(tdse_ctx* ctx, int32_t kind, int32_t slot) {
    if (!ctx) return fail(nullptr, TDSE_ERR_ARG, "ctx is NULL");
    if (kind == 1) {
        if (slot < 0 || slot >= (int)ctx->line.size() || !ctx->line[slot].live)
            return fail(ctx, TDSE_ERR_ARG, "bad Line slot");
        return TDSE_OK;  // a LineMesh always holds the reference g between launches
    }
    if (kind == 2) {
        if (slot < 0 || slot >= (int)ctx->cyl.size() || !ctx->cyl[slot].live) return fail(ctx, TDSE_ERR_ARG, "bad Cyl slot");
        HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
        int st[2] = {0, 0};  // step, phase
        char* base = reinterpret_cast<char*>(ctx->d_cyl + slot);
        HIP_TRY(ctx, hipMemcpy(&st[0], base + offsetof(CylSim, step), sizeof(int), hipMemcpyDeviceToHost));
        HIP_TRY(ctx, hipMemcpy(&st[1], base + offsetof(CylSim, phase), sizeof(int), hipMemcpyDeviceToHost));
        if (st[1] == 1) return TDSE_OK;
        return fail(ctx, TDSE_ERR_STATE,
                    "cylindrical state is between steps (explicit rho half applied); call tdse_set_hold before running "
                    "to stop at exact states");
    }
    if (kind != 0) return fail(ctx, TDSE_ERR_ARG, "unknown simulation kind");
    if (slot < 0 || slot >= (int)ctx->sh.size() || !ctx->sh[slot].live) return fail(ctx, TDSE_ERR_ARG, "bad SH slot");
    HIP_TRY(ctx, hipSetDevice(ctx->device));
    int rc;
    if (ctx->dirty && (rc = rebuild_tables(ctx))) return rc;
    HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
    int st[2] = {0, 0};  // step, phase
    char* base = reinterpret_cast<char*>(ctx->d_sh + slot);
    HIP_TRY(ctx, hipMemcpy(&st[0], base + offsetof(ShSim, step), sizeof(int), hipMemcpyDeviceToHost));
    HIP_TRY(ctx, hipMemcpy(&st[1], base + offsetof(ShSim, phase), sizeof(int), hipMemcpyDeviceToHost));
    const ShHost& H = ctx->sh[slot];
    if (st[1] == 1 || st[0] == 0 || st[0] > H.dev.N) return TDSE_OK;
    const int nw = H.wave_count;
    if (H.vel)
        hipLaunchKernelGGL((k_sh_lphase<false, true>), dim3((nw * TDSE_WAVE + 255) / 256), dim3(256), 0, ctx->stream,
                           ctx->d_sh, ctx->waves.ptr + H.wave_first, nw, ctx->d_clv, 1, ctx->d_sh);
    else
        hipLaunchKernelGGL((k_sh_lphase<false, false>), dim3((nw * TDSE_WAVE + 255) / 256), dim3(256), 0,
                           ctx->stream, ctx->d_sh, ctx->waves.ptr + H.wave_first, nw, ctx->d_cl, 1, ctx->d_sh);
    HIP_TRY(ctx, hipGetLastError());
    // the end-only L-phase wrote sh_state(n + 1): swap the buffers so the exact
    // state is sh_state(n) for the unchanged step counter
    ShSim& S = ctx->sh[slot].dev;
    std::swap(S.g, S.g2);
    const int one = 1;
    HIP_TRY(ctx, hipMemcpyAsync(base + offsetof(ShSim, g), &S.g, sizeof(S.g), hipMemcpyHostToDevice, ctx->stream));
    HIP_TRY(ctx, hipMemcpyAsync(base + offsetof(ShSim, g2), &S.g2, sizeof(S.g2), hipMemcpyHostToDevice, ctx->stream));
    HIP_TRY(ctx, hipMemcpyAsync(base + offsetof(ShSim, phase), &one, sizeof(int), hipMemcpyHostToDevice, ctx->stream));
    HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
    return TDSE_OK;
}

int tdse_last_run_ms(tdse_ctx* ctx, double* ms) {
    if (!ctx || !ms) return fail(ctx, TDSE_ERR_ARG, "NULL argument");
    *ms = ctx->last_run_ms;
    return TDSE_OK;
}

int tdse_profile(tdse_ctx* ctx, int32_t enable) {
    if (!ctx) return fail(nullptr, TDSE_ERR_ARG, "ctx is NULL");
    ctx->profiling = enable != 0;
    for (int i = 0; i < 6; ++i) {
        ctx->prof_ms[i] = 0.0;
        ctx->prof_n[i] = 0;
    }
    return TDSE_OK;
}

int tdse_profile_read(tdse_ctx* ctx, double* lphase_ms, int64_t* lphase_launches, double* rphase_ms,
                      int64_t* rphase_launches) {
    if (!ctx) return fail(nullptr, TDSE_ERR_ARG, "ctx is NULL");
    if (lphase_ms) *lphase_ms = ctx->prof_ms[0];
    if (lphase_launches) *lphase_launches = ctx->prof_n[0];
    if (rphase_ms) *rphase_ms = ctx->prof_ms[1];
    if (rphase_launches) *rphase_launches = ctx->prof_n[1];
    return TDSE_OK;
}

int tdse_profile_kernel(tdse_ctx* ctx, int32_t kernel, double* ms, int64_t* launches) {
    if (!ctx) return fail(nullptr, TDSE_ERR_ARG, "ctx is NULL");
    if (kernel < 0 || kernel > 5) return fail(ctx, TDSE_ERR_ARG, "kernel must be 0..5");
    if (ms) *ms = ctx->prof_ms[kernel];
    if (launches) *launches = ctx->prof_n[kernel];
    return TDSE_OK;
}

}  // extern "C"
