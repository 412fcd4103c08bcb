// common/splitk_host.h -- host side of the split-K launches, frozen into each delivery's
// kernel.hip after the kernels (it names k_splitk_reduce): the workspace a split-K row needs,
// where it comes from, and how many splits a row takes.
//
// A split-K row adds fp32 partial sums of its k ranges, [splits][M][N], in a workspace and reduces
// them with k_splitk_reduce on the same stream.  The workspace is either memory the caller hands
// over, or the delivery's pool: one buffer per (device, stream), allocated on first use and grown
// when a larger shape needs it, so calls on different streams stay independent.  A call is two
// kernels, and a stream orders kernels, not calls: the pool's buffer is leased, locked from before
// the first is enqueued until after the second, so that no other thread's partial sums land
// between them.

// Workspace of a split-K row.  `ptr`/`bytes`: device memory the caller hands over (may be
// null / 0), `shared` where calls on other streams take the same memory; `pool`: the row may take
// the delivery's per-(device, stream) pool instead; `need`: when set, the row only reports the
// bytes it needs (0 for rows without a workspace) and launches nothing.
struct Workspace {
  void* ptr = nullptr;
  size_t bytes = 0;
  bool pool = false;
  bool shared = false;
  size_t* need = nullptr;
};

// The workspace of one call, from workspace_for() until the call's last kernel is enqueued.  ptr is
// null where none could be had; `held` locks a pool buffer (nothing for the caller's memory).
struct Lease {
  float* ptr = nullptr;
  std::unique_lock<std::mutex> held;
};

// The pool: one buffer per (device, stream), grown on demand.  A buffer that a larger shape
// outgrows is retired, not freed: work already queued on the stream or a graph captured earlier
// may still use it, so it stays allocated until the process ends.  Sizes are whole powers of two
// from 1 MiB, so the retired buffers of a stream together stay below its current one.  Growing
// needs hipMalloc, which a stream under graph capture cannot take: there the pool returns
// hipErrorStreamCaptureUnsupported and the caller hands over its workspace instead (launch_with,
// or the C ABI's *_launch_ws entry points).  (The frozen file's preamble includes <map>, <mutex>,
// <utility> and <vector>.)
struct PoolBuffer {
  std::mutex busy;
  void* ptr = nullptr;
  size_t bytes = 0;
  std::vector<void*> retired;
};
inline Lease pool_lease(hipStream_t s, size_t bytes, hipError_t* err) {
  static std::mutex mu;
  static std::map<std::pair<int, hipStream_t>, PoolBuffer> pool;  // nodes keep their address
  Lease l;
  int dev = 0;
  if ((*err = hipGetDevice(&dev)) != hipSuccess) return l;
  PoolBuffer* e = nullptr;
  {
    std::lock_guard<std::mutex> lock(mu);
    e = &pool[std::make_pair(dev, s)];
  }
  std::unique_lock<std::mutex> held(e->busy);
  if (e->bytes < bytes) {
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    if ((*err = hipStreamIsCapturing(s, &cs)) != hipSuccess) return l;
    if (cs != hipStreamCaptureStatusNone) {
      *err = hipErrorStreamCaptureUnsupported;
      return l;
    }
    size_t size = (size_t)1 << 20;
    while (size < bytes) size *= 2;
    // another stream's capture, which would forbid this thread's hipMalloc, is none of its concern
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
    if ((*err = hipThreadExchangeStreamCaptureMode(&mode)) != hipSuccess) return l;
    void* q = nullptr;
    const hipError_t got = hipMalloc(&q, size);
    *err = hipThreadExchangeStreamCaptureMode(&mode);
    if (got != hipSuccess) {
      (void)hipGetLastError();  // the caller may go on without a workspace
      *err = hipErrorOutOfMemory;
      return l;
    }
    if (e->ptr) e->retired.push_back(e->ptr);
    e->ptr = q;
    e->bytes = size;
  }
  l.ptr = static_cast<float*>(e->ptr);
  l.held = std::move(held);
  return l;
}

// The workspace of a split-K launch: the caller's if it is large enough, else the pool's when the
// row may take it.  Null with *err set otherwise (hipErrorOutOfMemory: the caller's buffer is
// too small and no pool was allowed).
inline Lease workspace_for(const Workspace& w, size_t bytes, hipStream_t s, hipError_t* err) {
  *err = hipSuccess;
  if (w.pool && !(w.ptr && w.bytes >= bytes)) return pool_lease(s, bytes, err);
  Lease l;
  if (w.ptr && w.bytes >= bytes)
    l.ptr = static_cast<float*>(w.ptr);
  else
    *err = hipErrorOutOfMemory;
  return l;
}

// The workspace of a split that a row only gains by: its own path needs `own` bytes.  Where that is
// none, the call takes no memory that work on another stream may be using -- a `shared` workspace,
// the pool of a stream under capture (its graph may be replayed on any stream), the pool under
// hipStreamPerThread (one handle, a stream per thread) -- so that calls which need nothing share
// nothing.
inline Lease workspace_to_gain(const Workspace& w, size_t bytes, size_t own, hipStream_t s,
                               hipError_t* err) {
  if (own == 0) {
    const bool given = w.ptr && w.bytes >= bytes;
    bool refuse = given ? w.shared : w.pool && s == hipStreamPerThread;
    if (!given && w.pool && !refuse) {
      hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
      if (hipStreamIsCapturing(s, &cs) != hipSuccess) {
        (void)hipGetLastError();  // the caller goes on without a workspace
        refuse = true;
      }
      refuse = refuse || cs != hipStreamCaptureStatusNone;
    }
    if (refuse) {
      *err = hipErrorOutOfMemory;
      return Lease{};
    }
  }
  return workspace_for(w, bytes, s, err);
}

// Split count of a split-K row: the most splits such that tiles x splits stays within `slots`
// workgroups (one round of the part: a split count that spills into a second round makes every
// split of that round wait for it), each split keeping at least `minkt` k-tiles, and no split
// empty.  1 = no split.
inline int split_count(int tiles, int ktiles, int slots, int minkt) {
  if (slots <= 0 || minkt <= 0 || 2 * tiles > slots) return 1;
  int sp = slots / tiles;
  if (sp > ktiles / minkt) sp = ktiles / minkt;
  if (sp <= 1) return 1;
  const int per = (ktiles + sp - 1) / sp;
  return (ktiles + per - 1) / per;
}

// A plan picks, for one shape, the tile of the interleaved kernel and the split count with the
// least estimated time.  A table serves the rows up to m_max: microseconds per 1000 k of one round
// of a tile (one workgroup on each of the 256 CUs; per weight format), and what a round, a split
// (its second kernel) and a MB of partial sums (written and read) add.  The figures are fits to
// measured grids (100 .. 2200 workgroups; N = 1024 .. 34816, K = 2560 .. 17408) and order the
// alternatives only.  As times they are low: over random shapes at M > 64 with the weights from HBM
// splits take 1.16 times as long (median of 2054; 1.00 to 1.34 at the 5th and 95th percentile),
// unsplit tiles 1.09 times (of 2675; 0.91 to 1.67, the latter at short K) -- (200, 15360, 3840) fp16
// 42 us for 34, (2048, 2 x 17408, 5120) int8 620 for 501 -- for a round's rate depends on the clock
// under load and, below M = 256, on the HBM.
struct TileDims {
  int bm, bn, bk;
  bool splits;  // instantiated with split-K (the 256 x 256 tiles spill with it)
};
struct TileRate {
  int tile;
  double us[2];
};
struct PlanTable {
  int m_max;
  double round, split, mb;
  double weights;  // the least a million weights take (HBM), whatever the tile
  int n;
  TileRate rate[6];
};
struct TilePlan {
  int tile, splits;  // tile -1: none fits
  double us;
};
constexpr size_t kPlanWorkspace = (size_t)32 << 20;  // the allocation-free entry point's scratch

// The table of M rows (the last one has no bound).
inline const PlanTable& plan_table(const PlanTable* tabs, int M) {
  while (M > tabs->m_max) ++tabs;
  return *tabs;
}
inline double tile_us(const PlanTable& t, double rate, int bm, int bn, int bk, int M, int N, int K,
                      int splits) {
  const int ktiles = K / bk, per = (ktiles + splits - 1) / splits;
  const long wgs = (long)((M + bm - 1) / bm) * (N / bn) * splits;
  const double rounds = (double)((wgs + 255) / 256), hbm = t.weights * 1e-6 * N * K;
  double us = rounds * per * bk * rate * 1e-3;
  us = (us > hbm ? us : hbm) + rounds * t.round;
  return splits == 1 ? us : us + t.split + t.mb * 8e-6 * splits * M * N;
}
inline TilePlan plan_tiles(const TileDims* dims, const PlanTable* tabs, int f, int M, int N, int K,
                           bool split) {
  const PlanTable& t = plan_table(tabs, M);
  TilePlan best = {-1, 1, 0};
  for (int i = 0; i < t.n; ++i) {
    const TileDims& d = dims[t.rate[i].tile];
    if (N % d.bn || K % d.bk) continue;
    const int ktiles = K / d.bk;
    const long tiles = (long)((M + d.bm - 1) / d.bm) * (N / d.bn);
    for (int sp = 1; sp <= (split && d.splits ? 16 : 1); ++sp) {
      const int per = (ktiles + sp - 1) / sp;
      if (sp > 1 && (per * d.bk < 256 || tiles * sp > 512 ||
                     (size_t)sp * M * N * sizeof(float) > kPlanWorkspace))
        break;
      if ((ktiles + per - 1) / per != sp) continue;  // a split would be empty
      const double us = tile_us(t, t.rate[i].us[f], d.bm, d.bn, d.bk, M, N, K, sp);
      if (best.tile < 0 || us < best.us) best = {t.rate[i].tile, sp, us};
    }
  }
  return best;
}

// Launch of the split-K reduction: C = fp16_rn(sum over the splits of ws), in split order.
template <int UNROLL>
inline void run_reduce(const float* ws, int splits, int M, int N, _Float16* C, int ldc,
                       hipStream_t s) {
  const long work = (long)M * N / 4;
  hipLaunchKernelGGL(k_splitk_reduce<UNROLL>, dim3((unsigned)((work + 255) / 256)), dim3(256), 0, s,
                     ws, splits, M, N, C, ldc);
}
inline hipError_t launch_reduce(const float* ws, int splits, int M, int N, _Float16* C, int ldc,
                                hipStream_t s) {
  switch (splits) {  // every split's load in flight at once
    case 2: run_reduce<2>(ws, splits, M, N, C, ldc, s); break;
    case 3: run_reduce<3>(ws, splits, M, N, C, ldc, s); break;
    case 4: run_reduce<4>(ws, splits, M, N, C, ldc, s); break;
    case 5: run_reduce<5>(ws, splits, M, N, C, ldc, s); break;
    case 6: run_reduce<6>(ws, splits, M, N, C, ldc, s); break;
    case 7: run_reduce<7>(ws, splits, M, N, C, ldc, s); break;
    case 1: run_reduce<1>(ws, splits, M, N, C, ldc, s); break;
    default: run_reduce<8>(ws, splits, M, N, C, ldc, s);
  }
  return hipGetLastError();
}

// The same for the fused gate/up product: ws holds [S][M][2N] sums, the gate columns then the up
// columns.
inline hipError_t launch_reduce_gu(const float* ws, int splits, int M, int N, _Float16* C, int ldc,
                                   hipStream_t s) {
  const long work = (long)M * N / 4;
  const dim3 grid((unsigned)((work + 255) / 256)), blk(256);
  if (splits <= 2)
    hipLaunchKernelGGL(k_splitk_reduce_gu<2>, grid, blk, 0, s, ws, splits, M, N, C, ldc);
  else
    hipLaunchKernelGGL(k_splitk_reduce_gu<4>, grid, blk, 0, s, ws, splits, M, N, C, ldc);
  return hipGetLastError();
}
