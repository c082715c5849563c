// All layers of a decode step (ironcore/models/transformer.py:77-162, pre-LN) in one launch, for models so small that the
// launches of step_linear.hip are what a step waits for: GPT-2 small, fp32, batch 4 is 7 launches a layer of 5-6 us each, of
// which a product spends 2-3 us on the cold round trips to its weights, while all weights of a layer are 4.8 us of HBM.
//
//  * A layer is five kinds of task: projections (norm, bias, rotation), attention (append), output projection (residual),
//    up-projection (norm, bias, activation), down-projection (residual).  Tasks are numbered in that order, layer by layer.
//    A product's task is a tile of 64 bytes of columns; k is cut into splits, the last of which adds the others' sums in
//    order.  One task more per row norms the last layer's output.
//  * Every workgroup (one to a CU) goes through its tasks in ascending order: eight waves compute, four fetch the next
//    task's weights into LDS, which depends on nothing.  Some 2.4 tasks a layer fall on a CU, so a task's weights are on
//    their way while others run elsewhere.
//  * What tasks hand to each other goes through words in the workspace that are filled with kMissing before the launch:
//    a word that is something else is there.  Producers and consumers use relaxed atomics of device scope and nothing else:
//    no word's meaning depends on when another one becomes visible.  (A result that is bit for bit kMissing, a NaN, is
//    stored as another NaN.)
//  * Waits end whatever else runs on the GPU.  If all workgroups meet at the start (they are then all resident and stay so),
//    workgroup r takes the tasks r, r + workgroups, ...  If they do not within kMeetTicks (other streams hold CUs), tasks
//    are drawn from a counter: a task waits for tasks with lower numbers only, those are drawn before it by workgroups that
//    are running, and of the tasks drawn and not finished the lowest waits for nothing.  Either way is chosen once, by one
//    word.  (A ticket each time costs: 3.7 us from task to task over all CUs, 2.3 without.)  A wait that lasts for kMaxPolls
//    polls all the same (seconds) is given up: the words that it lacks are NaNs and make NaNs of what comes of them.  That is
//    known everywhere (kGaveUp) before any such word is handed on, and a row of K or V that may be one is not appended.
//
// Bound by the hand-over: from the last result of a phase to its arrival in all workgroups 1.5-2 us (past the L2s), five
// times a layer and once more for the splits of the down-projection, then 0.8-2 us for the phase itself; the launches
// it replaces are 2.8 us apart without any work.  GPT-2 small, fp32, batch 4, 12 layers: 517 -> 274 us a token; 128 + 64
// tokens by graph replay 36.0 -> 25.9 ms.
#include "decode_pair.h"
#include "ic_device.h"
#include "ic_internal.h"
#include "rope_device.h"
#include "step_common.h"
#include "../../include/ironcore_paged.h"

namespace ic {

using namespace step;
using namespace decode;

namespace {

constexpr uint32_t kMissing = 0xffffffffu;
constexpr uint64_t kMeetTicks = 3000;                    // of the 100 MHz counter
constexpr int kMaxPolls = 1 << 22;  // of a wait, unless the call says otherwise

enum Phase { kQkv = 0, kAttend = 1, kProj = 2, kUp = 3, kDown = 4, kPhases = 5 };

// The first words of the workspace: workgroups that have started, how tasks are dealt (0 open, 1 in turn, 2 drawn), the
// next task to draw, a wait was given up.  Each in a cache line of its own.
enum Control { kArrived = 0, kDealt = 32, kNext = 64, kGaveUp = 96, kControlWords = 128 };

struct StackKP {
  ic_step_layer layer[IC_STEP_STACK_LAYERS];
  const char *x;
  char *out, *norm_out;
  const char *last_weight, *last_bias;
  uint32_t *control;
  char *shared;           // the layers' words
  int64_t layer_bytes;    // of a layer
  int64_t at_att, at_mid, at_act, at_h, at_part;  // (the projections' rows lie first)
  int layers, m, d, f, n_up, q_cols, kv_cols, act, gated, last_norm;
  float last_eps;
  int first[kPhases + 1];  // first task of each phase of a layer, tasks of a layer
  int total;               // tasks of the launch
  int tiles_d, proj_splits, down_splits;
  DecodeKP dec;           // pools, query and output unset
  const int64_t *slots;
  const int32_t *positions;
  const float *cos_table, *sin_table;
  int64_t num_slots, table_rows;
  int gn, hd, must_draw;
  uint32_t poll_mask, max_polls;
  int32_t *status;
};
static_assert(sizeof(StackKP) <= 4096, "kernel arguments");

// The layers as the launch left them: an index that the compiler does not know would copy a by-value table to scratch.
typedef const __attribute__((address_space(4))) ic_step_layer LayerArgs;
__device__ __forceinline__ LayerArgs *layer_args() {
  static_assert(offsetof(StackKP, layer) == 0, "the layers come first");
  return (LayerArgs *)__builtin_amdgcn_kernarg_segment_ptr();
}

#define IC_INLINE __attribute__((always_inline))

// ---- words that tasks hand to each other -------------------------------------------------------

__device__ __forceinline__ uint32_t peek(const uint32_t *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ uint64_t peek8(const char *p) {
  return __hip_atomic_load(reinterpret_cast<const uint64_t *>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ bool there(uint64_t w) { return (uint32_t)w != kMissing && (uint32_t)(w >> 32) != kMissing; }
__device__ __forceinline__ uint32_t as_word(uint32_t w) { return w == kMissing ? 0x7fff7fffu : w; }

// Two neighbouring values: two words in fp32, one in the 16-bit types.
template <class E>
__device__ __forceinline__ void publish(char *at, float a, float b) {
  using T = typename E::type;
  if constexpr (sizeof(T) == 4) {
    const uint64_t w = (uint64_t)as_word(__builtin_bit_cast(uint32_t, b)) << 32 | as_word(__builtin_bit_cast(uint32_t, a));
    __hip_atomic_store(reinterpret_cast<uint64_t *>(at), w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  } else {
    const T lo = E::narrow(a), hi = E::narrow(b);
    const uint32_t w = (uint32_t)__builtin_bit_cast(uint16_t, hi) << 16 | __builtin_bit_cast(uint16_t, lo);
    __hip_atomic_store(reinterpret_cast<uint32_t *>(at), as_word(w), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

// A pause between two polls; true: give the wait up.
__device__ __forceinline__ bool pause(const StackKP &p, uint32_t &polls) {
  __builtin_amdgcn_s_sleep(1);
  if ((++polls & p.poll_mask) != 0) return false;
  const __attribute__((address_space(4))) StackKP *rare = (const __attribute__((address_space(4))) StackKP *)layer_args();
  asm volatile("" : "+s"(rare));  // (read here only: as arguments they would be kept in registers throughout)
  if (polls >= rare->max_polls) {
    int32_t *const status = rare->status;
    __hip_atomic_store(rare->control + kGaveUp, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (status != nullptr) __hip_atomic_store(status, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");  // before what this workgroup hands on from now
  }
  return peek(rare->control + kGaveUp) != 0;
}

// Two neighbouring values that a lane needs: as they are, and waited for (plain: a tensor from before the launch).
template <class E>
__device__ __forceinline__ uint64_t peek_pair(const char *at) {
  if constexpr (sizeof(typename E::type) == 4) return peek8(at);
  return peek(reinterpret_cast<const uint32_t *>(at));
}
template <class E>
__device__ __forceinline__ float2 take_pair(const StackKP &p, const char *at, bool plain, uint64_t w) {
  using T = typename E::type;
  uint32_t polls = 0;
  auto missing = [&] { return sizeof(T) == 4 ? !there(w) : (uint32_t)w == kMissing; };
  while (!plain && missing() && !pause(p, polls)) w = peek_pair<E>(at);
  if constexpr (sizeof(T) == 4)
    return make_float2(__builtin_bit_cast(float, (uint32_t)w), __builtin_bit_cast(float, (uint32_t)(w >> 32)));
  else
    return make_float2(static_cast<float>(__builtin_bit_cast(T, (uint16_t)w)),
                       static_cast<float>(__builtin_bit_cast(T, (uint16_t)(w >> 16))));
}

__device__ __forceinline__ Vec16 take16(const StackKP &p, const char *at) {
  uint32_t polls = 0;
  uint64_t a, b;
  do {
    a = peek8(at), b = peek8(at + 8);
  } while (!(there(a) && there(b)) && !pause(p, polls));
  return Vec16{{(uint32_t)a, (uint32_t)(a >> 32), (uint32_t)b, (uint32_t)(b >> 32)}};
}

// The attention task's view of the step's rows: published by the projections, rotated as they are stored.
template <class E, int HD, int GT>
struct StackRows {
  static constexpr bool kNew = true, kLate = true;
  static constexpr int EPL = E::EPL, ES = sizeof(typename E::type);
  const StackKP &p;
  const char *rows;  // [m][q | k | v]
  const int seq, kvh, lane, col;
  int64_t slot = -1;
  Vec16 own_k, own_v;
  __device__ __forceinline__ StackRows(const StackKP &p, const char *rows, int seq, int kvh, int lane)
      : p(p), rows(rows), seq(seq), kvh(kvh), lane(lane), col(lane % (HD / EPL)) {}
  __device__ __forceinline__ const char *at(int j, int column) const {
    return rows + ((int64_t)j * (p.q_cols + 2 * p.kv_cols) + column + col * EPL) * ES;
  }
  __device__ __forceinline__ Vec16 key(int j) const { return take16(p, at(j, p.q_cols + kvh * HD)); }
  __device__ __forceinline__ Vec16 value(int j) const { return take16(p, at(j, p.q_cols + p.kv_cols + kvh * HD)); }
  // Whether the pair's own row, which is there, may be appended.
  __device__ __forceinline__ bool sound() const { return peek(p.control + kGaveUp) == 0; }
  __device__ __forceinline__ void early() {
    slot = p.slots[lane < p.m ? lane : 0];
    if (lane >= p.m || slot >= p.num_slots) slot = -1;
  }
  __device__ __forceinline__ void queries(Vec16 *qreg) {
    uint64_t w[GT + 2][2];
    uint32_t polls = 0;
    bool ok;
    do {
#pragma unroll
      for (int g = 0; g < GT + 2; ++g) {
        const int column = g < GT ? (kvh * p.dec.group + (g < p.dec.group ? g : p.dec.group - 1)) * HD
                                  : p.q_cols + (g - GT) * p.kv_cols + kvh * HD;
        w[g][0] = peek8(at(seq, column)), w[g][1] = peek8(at(seq, column) + 8);
      }
      ok = true;
#pragma unroll
      for (int g = 0; g < GT + 2; ++g) ok = ok && there(w[g][0]) && there(w[g][1]);
    } while (!__all(ok) && !pause(p, polls));
    auto vec = [&](int g) {
      return Vec16{{(uint32_t)w[g][0], (uint32_t)(w[g][0] >> 32), (uint32_t)w[g][1], (uint32_t)(w[g][1] >> 32)}};
    };
#pragma unroll
    for (int g = 0; g < GT; ++g) qreg[g] = vec(g);
    own_k = vec(GT), own_v = vec(GT + 1);
  }
};

// Counters in LDS by which the waves of a workgroup wait for each other.  Not s_barrier: the loaders would have to take part,
// and while a loader's requests fill the CU's queue it takes them a microsecond to get from one barrier to the next.
__device__ __forceinline__ void count_up(uint32_t *counter, int lane) {
  asm volatile("" ::: "memory");  // (LDS instructions of a wave are carried out in order)
  if (lane == 0) __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ void wait_count(const uint32_t *counter, uint32_t count) {
  while ((int)(__builtin_amdgcn_readfirstlane(__hip_atomic_load(counter, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP)) -
               count) < 0)
    __builtin_amdgcn_s_sleep(0);
  asm volatile("" ::: "memory");
}

constexpr int kLoaders = 4;  // waves that fetch weights (half of the product's: see fetch)
constexpr int kStackThreads = kStepThreads + kLoaders * kWave;

struct Task {
  int layer, phase, index;  // (phase kPhases: a row of the last norm; kPhases + 1: no task)
};

// (No index into the arguments that the compiler does not know: they would go through scratch.)
__device__ __forceinline__ Task task_of(const StackKP &p, int task) {
  const int per_layer = p.first[kPhases];
  const int layer = task / per_layer, at = task - layer * per_layer;
  if (task < 0 || task >= p.total) return Task{0, kPhases + 1, 0};
  if (layer >= p.layers) return Task{layer, kPhases, at};
  if (at < p.first[kAttend]) return Task{layer, kQkv, at};
  if (at < p.first[kProj]) return Task{layer, kAttend, at - p.first[kAttend]};
  if (at < p.first[kUp]) return Task{layer, kProj, at - p.first[kProj]};
  if (at < p.first[kDown]) return Task{layer, kUp, at - p.first[kUp]};
  return Task{layer, kDown, at - p.first[kDown]};
}

// Tile and split of a product's task.
template <int TN>
struct Tile {
  int mat, n, n0, half, split;  // second matrix of the projections; columns of the matrix; first of the tile; gated: its half
  __device__ __forceinline__ Tile(const StackKP &p, int phase, int index) {
    mat = 0, split = 0, half = 0, n = p.d;
    if (phase == kQkv) {
      const int tiles0 = p.q_cols / TN;
      mat = index >= tiles0;
      index -= mat ? tiles0 : 0;
      n = mat ? 2 * p.kv_cols : p.q_cols;
    } else if (phase == kUp) {
      n = p.n_up;
      half = p.gated ? n / 2 : 0;
    } else {
      split = index / p.tiles_d;
      index -= split * p.tiles_d;
    }
    n0 = index * (half ? TN / 2 : TN);
  }
};

template <class M, int HD, int GT, int S>
struct Stack {
  using E = typename M::E;
  using T = typename E::type;
  static constexpr int NB = 4 / sizeof(T);  // 64 bytes of columns: 16 words of 1 or 2 values
  using Sh = Shape<M, NB>;
  static constexpr int KR = Sh::KR, ES = Sh::ES, TN = Sh::TN, PITCH = Sh::PITCH;
  static constexpr int STEP_BYTES = Sh::STEP * 64, WAVE_BYTES = S * STEP_BYTES, NORM_BYTES = S * kStepWaves * 64;
  static constexpr int ROW_PITCH = NORM_BYTES + 64;  // of the rows of x: four rows by four chunks find 64 banks
  // Weights of a task and of its norm.  Once the weights are in registers, the rows of x go where they were; an attention
  // task, which has neither, uses the whole.
  struct Slot {
    union {
      char w[kStepWaves][WAVE_BYTES];
      char x[16][ROW_PITCH];
      PairShared<HD, GT> pair;
    };
    char gain[NORM_BYTES], shift[NORM_BYTES];
    char bias[1024];  // of the tile: 64 bytes
  };
  struct Shared {
    Slot slot[2];
    float sum[kStepWaves][16 * PITCH];
    float2 stat[kStepWaves][16];
    int task[2];
    uint32_t done, landed, drawn;  // barriers of the product's waves, tasks whose weights are there, tasks drawn
  };
  static_assert(sizeof(Shared) <= 160 * 1024, "LDS of a CU");
  const StackKP &p;
  Shared &sh;
  const int thread, lane, wave, c, g;
  // fp32, up to four rows: 4x4 products, a block of which has four columns and the k of one lane group, with nothing
  // computed for rows that are not there (16x16 products: 0.7 us more a task).
  const bool few;
  const int xrow;  // the lane's row of x
  uint32_t &passed;  // what `done` comes to at the last barrier
  const int64_t angle;  // first element of the thread's row (of the projections' sums) in the rotary tables

  // (`thread` is threadIdx.x as a value that the compiler does not know from one task to the next: it would keep every
  // lane's addresses for all kinds of task in registers, and those in scratch.)
  __device__ __forceinline__ Stack(const StackKP &p, Shared &sh, int thread, uint32_t &passed, int64_t angle)
      : p(p), sh(sh), thread(thread), lane(thread & (kWave - 1)),
        wave(__builtin_amdgcn_readfirstlane(thread / kWave)), c(lane & 15), g(lane >> 4),
        few(sizeof(T) == 4 && p.m <= 4), xrow(few ? c & 3 : c), passed(passed), angle(angle) {}

  // Barrier of the product's waves.
  __device__ __forceinline__ void barrier() const {
    passed += kStepWaves;
    count_up(&sh.done, lane);
    wait_count(&sh.done, passed);
  }
  __device__ __forceinline__ char *words(int layer) const { return p.shared + layer * p.layer_bytes; }
  // The steps of wave v: first + 8 i, those past the end of a column load the last one's weights and zeros of x.
  __device__ __forceinline__ int first_step(int split, int v) const { return split * S * kStepWaves + v; }

  // (loaders) Half of a task's weights on their way into a slot (those of four waves; with the first half the norm's and the
  // bias), 1 KiB of LDS an instruction: 16 rows of 64 bytes.  Row r of lane
  // group g lies at (4 r + g) * 64, so that the lanes that read it find 64 banks.
  __device__ __forceinline__ void fetch(const Task &task, Slot &slot, int half) const {
    if (task.phase >= kPhases || task.phase == kAttend) return;
    const Tile<TN> t(p, task.phase, task.index);
    LayerArgs &w = layer_args()[task.layer];
    const char *matrix = (const char *)(task.phase == kQkv ? (t.mat ? w.kv_weight : w.q_weight)
                                        : task.phase == kProj ? w.proj_weight : task.phase == kUp ? w.up_weight : w.down_weight);
    const int k = task.phase == kProj ? p.q_cols : task.phase == kDown ? p.f : p.d;
    const int steps = k * ES / 64, chunk = lane & 3;
    const uint32_t pitch = (uint32_t)t.n * ES;
    const uint32_t at = (uint32_t)((lane >> 2 & 3) * KR + (lane >> 4)) * pitch +
                        (t.half ? (uint32_t)(t.n0 + (chunk >> 1) * t.half) * ES + (chunk & 1) * 16
                                : (uint32_t)t.n0 * ES + chunk * 16);
    const int loader = wave - kStepWaves;
    typedef __attribute__((address_space(1))) void Global;
    typedef __attribute__((address_space(3))) void Local;
    auto copy = [&](const char *from, char *to) IC_INLINE {
      __builtin_amdgcn_global_load_lds((Global *)from, (Local *)to, 16, 0, 0);
    };
#pragma unroll
    for (int i = 0; i < S; ++i) {
      const int v = loader + half * kLoaders;
      const int step = first_step(t.split, v) + i * kStepWaves;
      const char *from = matrix + (int64_t)(step < steps ? step : steps - 1) * Sh::STEP * pitch + at;
#pragma unroll
      for (int j = 0; j < KR / 4; ++j) copy(from + j * 4 * (uint64_t)pitch, slot.w[v] + i * STEP_BYTES + j * 1024);
    }
    if (half > 0) return;
    const char *bias = (const char *)(task.phase == kQkv ? (t.mat ? w.kv_bias : w.q_bias)
                                      : task.phase == kProj ? w.proj_bias : task.phase == kUp ? w.up_bias : w.down_bias);
    if (bias != nullptr && loader == 0)
      copy(bias + (t.half ? (t.n0 + (chunk >> 1) * t.half) * ES + (chunk & 1) * 16 : t.n0 * ES + chunk * 16), slot.bias);
    if (task.phase == kQkv || task.phase == kUp) {
      const char *gains = (const char *)(task.phase == kQkv ? w.input_norm_weight : w.post_norm_weight);
      const char *shifts = (const char *)(task.phase == kQkv ? w.input_norm_bias : w.post_norm_bias);
      for (int i = loader; i < NORM_BYTES / 1024; i += kLoaders) {
        const int byte = i * 1024 + lane * 16, end = p.d * ES - 16;
        copy(gains + (byte < end ? byte : end), slot.gain + i * 1024);
        if (shifts != nullptr) copy(shifts + (byte < end ? byte : end), slot.shift + i * 1024);
      }
    }
  }

  // The task's part of the rows `from` [m][k], waited for unless they are `plain`, into LDS: neighbouring lanes take
  // neighbouring words, since each of these requests goes past the L2s.  (Straight into the lanes of the product they were
  // eight times as many, and a task 4 us behind the one before it, not 2.)
  // The wave's rows row, row + 8, ..., of each the 512-byte pieces begin .. begin + N - 1.
  // `residual` (or null): two values more that the thread needs, which are there by then.
  template <int ROWS, int N>
  __device__ __forceinline__ void take_words(const char *from, int row_bytes, int part, int row, int begin, bool plain,
                                             Slot &slot, const char *residual, uint64_t &res_word) const {
    if (row >= p.m) {
      if (residual != nullptr) res_word = peek_pair<E>(residual);
      return;
    }
    const bool second = ROWS > 1 && row + 8 < p.m;
    auto offset = [&](int i) IC_INLINE {  // (past the end of a short last part: its last word)
      const int byte = (begin + i) * 512 + lane * 8;
      return byte < part ? byte : part - 8;
    };
    const char *const at = from + (int64_t)row * row_bytes;
    const int64_t step = second ? 8 * (int64_t)row_bytes : 0;
    uint32_t polls = 0;
    uint64_t w[ROWS][N];
    for (;;) {
      bool ok = true;
#pragma unroll
      for (int r = 0; r < ROWS; ++r)
#pragma unroll
        for (int i = 0; i < N; ++i) w[r][i] = peek8(at + r * step + offset(i));
      if (residual != nullptr) res_word = peek_pair<E>(residual);
#pragma unroll
      for (int r = 0; r < ROWS; ++r)
#pragma unroll
        for (int i = 0; i < N; ++i) ok = ok && there(w[r][i]);
      if (plain || __all(ok) || pause(p, polls)) break;
    }
#pragma unroll
    for (int r = 0; r < ROWS; ++r)
#pragma unroll
      for (int i = 0; i < N; ++i)
        if (r == 0 || second) *reinterpret_cast<uint64_t *>(slot.x[row + 8 * r] + (begin + i) * 512 + lane * 8) = w[r][i];
  }
  __device__ __forceinline__ void take_rows(const char *from, int k, int split, bool plain, Slot &slot, Vec16 (&xv)[S],
                                            const char *residual, uint64_t &res_word) const {
    const int row_bytes = k * ES, before = split * NORM_BYTES;
    const int part = row_bytes - before < NORM_BYTES ? row_bytes - before : NORM_BYTES;
    if (p.m <= 4)  // two waves to a row
      take_words<1, S / 2>(from + before, row_bytes, part, wave & 3, (wave >> 2) * (S / 2), plain, slot, residual, res_word);
    else
      take_words<2, S>(from + before, row_bytes, part, wave, 0, plain, slot, residual, res_word);
    barrier();
    const bool wanted = xrow < p.m;
#pragma unroll
    for (int i = 0; i < S; ++i) {
      const int byte = (wave + i * kStepWaves) * 64;
      const bool in = wanted && byte < part;
      const Vec16 v = load16(slot.x[wanted ? xrow : 0] + (byte < part ? byte : 0) + g * 16);
#pragma unroll
      for (int e = 0; e < 4; ++e) xv[i].w[e] = in ? v.w[e] : 0u;
    }
  }

  // The rows' norm in place.  Mean and squares of a row: each lane's own by two passes over its registers, then merged
  // (counts, means, squares about them), which loses nothing to cancellation and needs one barrier.
  __device__ __forceinline__ void norm_rows(Vec16 (&xv)[S], const Slot &slot, bool shifted, bool centered, float eps) const {
    const int steps = p.d * ES / 64;
    auto steps_of = [&](int v) IC_INLINE { return (steps - v + kStepWaves - 1) / kStepWaves; };
    const int mine = steps_of(wave);
    const float own = (float)(mine * KR);
    float mean = 0.f, squares = 0.f, f[KR];
    if (centered) {
#pragma unroll
      for (int i = 0; i < S; ++i) {
        E::widen(xv[i], f);
#pragma unroll
        for (int e = 0; e < KR; ++e) mean += f[e];  // (steps past the last are zeros)
      }
      mean = mine > 0 ? mean / own : 0.f;
    }
#pragma unroll
    for (int i = 0; i < S; ++i) {
      E::widen(xv[i], f);
      float part = 0.f;
#pragma unroll
      for (int e = 0; e < KR; ++e) part = __builtin_fmaf(f[e] - mean, f[e] - mean, part);
      squares += i < mine ? part : 0.f;
    }
#pragma unroll
    for (int off = 16; off < kWave; off <<= 1) {  // (equal counts)
      const float other = __shfl_xor(mean, off, kWave), by = mean - other, count = own * (float)(off / 16);
      squares += __shfl_xor(squares, off, kWave) + by * by * count * 0.5f;
      mean = 0.5f * (mean + other);
    }
    if (g == 0) sh.stat[wave][c] = make_float2(mean, squares);
    barrier();
    float2 part[kStepWaves];
    float center = 0.f, total = 0.f;
#pragma unroll
    for (int i = 0; i < kStepWaves; ++i) {
      part[i] = sh.stat[i][c];
      center += part[i].x * (float)steps_of(i);
    }
    center /= (float)steps;
#pragma unroll
    for (int i = 0; i < kStepWaves; ++i) {
      const float by = part[i].x - center;
      total += part[i].y + by * by * (float)(steps_of(i) * Sh::STEP);
    }
    const float scale = 1.f / sqrtf(total / (float)p.d + eps);
#pragma unroll
    for (int i = 0; i < S; ++i) {
      float gv[KR], sv[KR];
      E::widen(xv[i], f);
      const int at = (wave + i * kStepWaves) * 64 + g * 16;
      E::widen(load16(slot.gain + at), gv);
      E::widen(shifted ? load16(slot.shift + at) : Vec16{{0u, 0u, 0u, 0u}}, sv);
#pragma unroll
      for (int e = 0; e < KR; ++e) f[e] = i < mine ? (f[e] - center) * scale * gv[e] + sv[e] : 0.f;
      if constexpr (sizeof(T) == 4) {
#pragma unroll
        for (int e = 0; e < 4; ++e) xv[i].w[e] = __builtin_bit_cast(uint32_t, f[e]);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const T lo = E::narrow(f[2 * e]), hi = E::narrow(f[2 * e + 1]);
          xv[i].w[e] = (uint32_t)__builtin_bit_cast(uint16_t, hi) << 16 | __builtin_bit_cast(uint16_t, lo);
        }
      }
    }
  }

  // The wave's sums of the tile, [row of x][column] in LDS, over its first `used` steps (those past the end of a column hold
  // other rows' weights: with zeros of x they add nothing, but a NaN if a weight is infinite).
  __device__ __forceinline__ void multiply_block(const Words<1> (&wv)[S][KR], const Vec16 (&xv)[S], int used) const {
    float *const sums = sh.sum[wave];
    f32x4_t acc[NB][1];
#pragma unroll
    for (int j = 0; j < NB; ++j) acc[j][0] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    if (few) {
      if constexpr (sizeof(T) == 4) {
#pragma unroll
        for (int i = 0; i < S; ++i) {
          if (i >= used) break;
#pragma unroll
          for (int r = 0; r < KR; ++r)
            acc[0][0] = __builtin_amdgcn_mfma_f32_4x4x1f32(__builtin_bit_cast(float, wv[i][r].w[0]),
                                                           __builtin_bit_cast(float, xv[i].w[r]), acc[0][0], 0, 0, 0);
        }
        // lane (c, g): columns 4 * (c / 4) + r of row c % 4, the k of lane group g
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          acc[0][0][r] += __shfl_xor(acc[0][0][r], 16, kWave);
          acc[0][0][r] += __shfl_xor(acc[0][0][r], 32, kWave);
        }
        if (g == 0)
          *reinterpret_cast<float4 *>(sums + (c & 3) * PITCH + (c >> 2) * 4) =
              make_float4(acc[0][0][0], acc[0][0][1], acc[0][0][2], acc[0][0][3]);
      }
      return;
    }
#pragma unroll
    for (int i = 0; i < S; ++i) {
      if (i >= used) break;
      const Vec16 x[1] = {xv[i]};
      if constexpr (sizeof(T) == 4) {  // (a step's own sum: one chain over all would round as often as it has products)
        f32x4_t step[NB][1] = {{{0.f, 0.f, 0.f, 0.f}}};
        multiply<M, 1, NB>(wv[i], x, step);
        acc[0][0] += step[0][0];
      } else {
        multiply<M, 1, NB>(wv[i], x, acc);
      }
    }
    float *to = sums + c * PITCH + g * 4 * NB;
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int j = 0; j < NB; ++j) to[r * NB + j] = acc[j][0][r];
  }

  // Two columns of a row, all waves together.
  __device__ __forceinline__ float2 total(int row, int column) const {
    float2 sum = make_float2(0.f, 0.f);
#pragma unroll
    for (int v = 0; v < kStepWaves; ++v) {
      const float2 s = *reinterpret_cast<const float2 *>(sh.sum[v] + row * PITCH + column);
      sum.x += s.x, sum.y += s.y;
    }
    return sum;
  }

  template <int PHASE>
  __device__ __forceinline__ void run_product(int layer, int index, Slot &slot) const {
    constexpr bool kNormed = PHASE == kQkv || PHASE == kUp;
    const Tile<TN> t(p, PHASE, index);
    LayerArgs &w = layer_args()[layer];
    char *const mine_words = words(layer);
    const bool plain = layer == 0;  // the hidden rows are the call's
    const char *hidden = plain ? p.x : words(layer - 1) + p.at_h;
    // ---- everything that the end needs, before the wait ------------------------------------------
    // a thread takes two columns of one row
    const int cols = PHASE == kUp && t.half ? TN / 2 : TN;
    const int at = 2 * (thread & (cols / 2 - 1)), row = thread / (cols / 2);
    const bool mine = row < p.m;
    const int col = t.n0 + at;
    float bias_a = 0.f, bias_b = 0.f, gate_a = 0.f, gate_b = 0.f, turn_cos = 1.f, turn_sin = 0.f;
    char *to = nullptr;              // the result
    char *part = nullptr;            // partial sums of splits, this thread's of the first one
    const char *residual = nullptr;
    uint64_t res_word = kMissing;
    const int splits = PHASE == kProj ? p.proj_splits : PHASE == kDown ? p.down_splits : 1;
    const bool last = t.split + 1 == splits;
    const int64_t part_pitch = (int64_t)p.m * p.d * 4;
    bool turned = false;
    if (mine) {
      if ((PHASE == kQkv ? (t.mat ? w.kv_bias : w.q_bias) : PHASE == kProj ? w.proj_bias : PHASE == kUp ? w.up_bias : w.down_bias) !=
          nullptr) {
        const T *bias = reinterpret_cast<const T *>(slot.bias);
        bias_a = static_cast<float>(bias[at]), bias_b = static_cast<float>(bias[at + 1]);
        if (PHASE == kUp && t.half)
          gate_a = static_cast<float>(bias[TN / 2 + at]), gate_b = static_cast<float>(bias[TN / 2 + at + 1]);
      }
      if constexpr (PHASE == kQkv) {
        const int all = (t.mat ? p.q_cols : 0) + col;  // of [q | k | v]
        to = mine_words + ((int64_t)row * (p.q_cols + 2 * p.kv_cols) + all) * ES;
        turned = p.cos_table != nullptr && all < p.q_cols + p.kv_cols;
        if (turned) {
          const int64_t from = angle + (all & (HD - 1)) / 2;
          turn_cos = p.cos_table[from], turn_sin = p.sin_table[from];
        }
      } else if constexpr (PHASE == kUp) {
        to = mine_words + p.at_act + ((int64_t)row * p.f + col) * ES;
      } else {
        const int64_t offset = ((int64_t)row * p.d + col) * ES;
        to = mine_words + (PHASE == kProj ? p.at_mid : p.at_h) + offset;
        part = mine_words + p.at_part + (PHASE == kDown ? (p.proj_splits - 1) * part_pitch : 0) + ((int64_t)row * p.d + col) * 4;
        residual = (PHASE == kProj ? hidden : mine_words + p.at_mid) + offset;
      }
    }
    bool centered = false, shifted = false;
    float eps = 0.f;
    int act = PHASE == kUp ? p.act : 0;
    if constexpr (kNormed) {
      shifted = (PHASE == kQkv ? w.input_norm_bias : w.post_norm_bias) != nullptr;
      centered = (PHASE == kQkv ? w.input_norm : w.post_norm) == IC_NORM_LAYER;
      eps = PHASE == kQkv ? w.input_norm_eps : w.post_norm_eps;
      asm volatile("" : "+s"(eps), "+s"(act));
    }
    Words<1> wv[S][KR];
#pragma unroll
    for (int i = 0; i < S; ++i)
#pragma unroll
      for (int r = 0; r < KR; ++r)
        wv[i][r] = *reinterpret_cast<const Words<1> *>(slot.w[wave] + i * STEP_BYTES + (r * 4 + g) * 64 + c * 4);
    barrier();  // (the rows of x go where the weights are)
    // ---- the product -----------------------------------------------------------------------------
    Vec16 xv[S];
    const int k = PHASE == kProj ? p.q_cols : PHASE == kDown ? p.f : p.d;
    take_rows(PHASE == kQkv ? hidden : mine_words + (PHASE == kProj ? p.at_att : PHASE == kUp ? p.at_mid : p.at_act), k, t.split, PHASE == kQkv && plain, slot, xv, last ? residual : nullptr,
              res_word);
    if constexpr (kNormed) norm_rows(xv, slot, shifted, centered, eps);
    multiply_block(wv, xv, (k * ES / 64 - first_step(t.split, wave) + kStepWaves - 1) / kStepWaves);
    barrier();
    if (!mine) return;
    float2 v = total(row, at);
    if constexpr (PHASE == kProj || PHASE == kDown) {
      if (!last) {
        publish<F32>(part + t.split * part_pitch, v.x, v.y);
        return;
      }
      float2 sum = make_float2(0.f, 0.f);
      for (int s = 0; s + 1 < splits; ++s) {
        const float2 other = take_pair<F32>(p, part + s * part_pitch, false, peek8(part + s * part_pitch));
        sum.x += other.x, sum.y += other.y;
      }
      const float2 res = take_pair<E>(p, residual, PHASE == kProj && plain, res_word);
      publish<E>(to, sum.x + v.x + bias_a + res.x, sum.y + v.y + bias_b + res.y);
      return;
    }
    v.x += bias_a, v.y += bias_b;
    if constexpr (PHASE == kUp) {
      if (t.half) {
        float2 gate = total(row, TN / 2 + at);
        gate.x += gate_a, gate.y += gate_b;
        if (act == IC_ACT_SWIGLU)
          v.x = v.x * sigmoid(v.x) * gate.x, v.y = v.y * sigmoid(v.y) * gate.y;
        else
          v.x *= sigmoid(gate.x), v.y *= sigmoid(gate.y);
      } else {
        v.x = activate(act, v.x), v.y = activate(act, v.y);
      }
    }
    if (PHASE == kQkv && turned) rotate_pair(v.x, v.y, turn_cos, turn_sin, v.x, v.y);
    publish<E>(to, v.x, v.y);
  }

  __device__ __forceinline__ void run_attention(int layer, int index, Slot &slot) const {
    const int seq = index / p.gn, kvh = index - seq * p.gn;
    StackRows<E, HD, GT> rows(p, words(layer), seq, kvh, lane);
    char *out = words(layer) + p.at_att + ((int64_t)seq * p.q_cols + kvh * p.dec.group * HD) * ES;
    const int tiles = walk_pair<E, HD, GT>(p.dec, (const char *)layer_args()[layer].k_pool,
                                           (const char *)layer_args()[layer].v_pool, seq, kvh, thread, slot.pair, rows);
    barrier();
    const int o = 2 * thread;
    if (o < p.dec.group * HD)
      publish<E>(out + o * ES, tiles == 0 ? 0.f : pair_value(slot.pair, o / HD, o % HD),
                 tiles == 0 ? 0.f : pair_value(slot.pair, o / HD, o % HD + 1));
  }

  // A row of the last layer's output and its norm, 4 bytes a thread at a time.
  __device__ __forceinline__ void run_last(int row) const {
    constexpr int PER = 4 / sizeof(T), ITER = 2;
    const int n = p.d * ES / 4;
    const uint32_t *from = reinterpret_cast<const uint32_t *>(words(p.layers - 1) + p.at_h + (int64_t)row * p.d * ES);
    float v[ITER][PER];
    float sum = 0.f;
    auto widen = [&](uint32_t w, float *to) IC_INLINE {
      if constexpr (PER == 1) {
        to[0] = __builtin_bit_cast(float, w);
      } else {
        to[0] = static_cast<float>(__builtin_bit_cast(T, (uint16_t)w));
        to[1] = static_cast<float>(__builtin_bit_cast(T, (uint16_t)(w >> 16)));
      }
    };
#pragma unroll
    for (int i = 0; i < ITER; ++i) {
      const int at = i * kStepThreads + thread;
      uint32_t word = 0, polls = 0;
      if (at < n)
        do {
          word = peek(from + at);
        } while (word == kMissing && !pause(p, polls));
      widen(word, v[i]);
#pragma unroll
      for (int e = 0; e < PER; ++e) sum += v[i][e];
      if (at < n && p.out != nullptr) reinterpret_cast<uint32_t *>(p.out)[(int64_t)row * n + at] = word;
    }
    if (p.last_norm == IC_NORM_NONE) return;
    auto over_row = [&](float part, int buffer) IC_INLINE {
      part = group_sum<kWave>(part);
      if (lane == 0) sh.stat[wave][buffer].x = part;
      barrier();
      float total = 0.f;
#pragma unroll
      for (int i = 0; i < kStepWaves; ++i) total += sh.stat[i][buffer].x;
      return total;
    };
    const float inv_n = 1.f / (float)p.d;
    const float mean = p.last_norm == IC_NORM_LAYER ? over_row(sum, 0) * inv_n : 0.f;
    float squares = 0.f;
#pragma unroll
    for (int i = 0; i < ITER; ++i)
      if (i * kStepThreads + thread < n)
#pragma unroll
        for (int e = 0; e < PER; ++e) squares = __builtin_fmaf(v[i][e] - mean, v[i][e] - mean, squares);
    const float scale = 1.f / sqrtf(over_row(squares, 1) * inv_n + p.last_eps);
#pragma unroll
    for (int i = 0; i < ITER; ++i) {
      const int at = i * kStepThreads + thread;
      if (at >= n) continue;
      float gv[PER], sv[PER] = {};
      widen(reinterpret_cast<const uint32_t *>(p.last_weight)[at], gv);
      if (p.last_bias != nullptr) widen(reinterpret_cast<const uint32_t *>(p.last_bias)[at], sv);
      T *to = reinterpret_cast<T *>(p.norm_out) + (int64_t)row * p.d + at * PER;
#pragma unroll
      for (int e = 0; e < PER; ++e) to[e] = E::narrow((v[i][e] - mean) * scale * gv[e] + sv[e]);
    }
  }
};

template <class M, int HD, int GT, int S>
__global__ __launch_bounds__(kStackThreads) void step_stack_kernel(const StackKP p) {
  using K = Stack<M, HD, GT, S>;
  __shared__ __attribute__((aligned(1024))) typename K::Shared sh;
  const int lane = threadIdx.x & (kWave - 1);
  const bool loads = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave) >= kStepWaves;
  // Tasks two by two go round the XCDs: neighbours share the cache lines of W.
  const int b = blockIdx.x;
  int task = gridDim.x % 16 == 0 ? (b / 16) * 16 + (b % kXcds) * 2 + (b / kXcds) % 2 : b;
  Task now = task_of(p, task);
  uint32_t passed = 0, rounds = 0;
  if (loads) {
    const K kernel(p, sh, threadIdx.x, passed, 0);
    kernel.fetch(now, sh.slot[0], 0);
    kernel.fetch(now, sh.slot[0], 1);
  }
  int64_t angle = 0;
  if (const int row = threadIdx.x / (K::TN / 2); p.cos_table != nullptr && row < p.m) {
    const int64_t pos = p.positions[row];
    angle = (pos < 0 ? 0 : pos >= p.table_rows ? p.table_rows - 1 : pos) * (HD / 2);
  }
  // ---- how tasks are dealt ---------------------------------------------------------------------
  if (threadIdx.x == 0) {
    sh.done = sh.landed = sh.drawn = 0;
    uint32_t *const dealt = p.control + kDealt;
    uint32_t open = 0;
    const uint32_t before = __hip_atomic_fetch_add(p.control + kArrived, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (before + 1 == gridDim.x && !p.must_draw)
      __hip_atomic_compare_exchange_strong(dealt, &open, 1u, __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const uint64_t start = wall_clock64();
    uint32_t how;
    while ((how = peek(dealt)) == 0) {
      open = 0;
      if (p.must_draw || wall_clock64() - start > kMeetTicks)
        __hip_atomic_compare_exchange_strong(dealt, &open, 2u, __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    sh.task[1] = (int)how;
  }
  __syncthreads();
  const bool draw = __builtin_amdgcn_readfirstlane(sh.task[1]) == 2;
  if (draw) task = -1, now = task_of(p, -1);  // (no task yet; the first one's weights come with the next round)
  __syncthreads();
  for (int turn = 0;; turn ^= 1) {  // (the slot of `now`)
    ++rounds;
    int next = task + (int)gridDim.x;
    if (draw) {
      if (threadIdx.x == 0)
        sh.task[turn] = (int)__hip_atomic_fetch_add(p.control + kNext, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (threadIdx.x < kWave) count_up(&sh.drawn, lane);
      wait_count(&sh.drawn, rounds);
      next = __builtin_amdgcn_readfirstlane(sh.task[turn]);
    }
    if (task >= p.total) break;
    const Task then = task_of(p, next);
    int thread = threadIdx.x;
    asm volatile("" : "+v"(thread));
    const K kernel(p, sh, thread, passed, angle);
    typename K::Slot &slot = sh.slot[turn];
    if (loads) {
      // The loaders see this task's weights land.  The next one's, whose slot nobody reads any more, they ask for once this
      // one's input is there, and the second half once it has ended: a CU's requests are answered in turn, and polls and
      // results would wait behind 48 KiB of weights.  (GPT-2 small as below: all before the polls 30.3 ms, all with the input
      // there 26.1, all at the end 28.4, half and half 25.9.)
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      count_up(&sh.landed, lane);
      const int last_norm = p.last_norm;
      const int before = now.phase == kAttend ? 1 : now.phase < kPhases ? 2 : 0;  // barriers up to there, and after it
      const int after = now.phase == kQkv || now.phase == kUp ? 3 : now.phase == kAttend ? 1 : now.phase < kPhases ? 2
                        : now.phase > kPhases ? 1 : last_norm == IC_NORM_LAYER ? 3 : last_norm == IC_NORM_RMS ? 2 : 1;
      wait_count(&sh.done, passed + before * kStepWaves);
      kernel.fetch(then, sh.slot[turn ^ 1], 0);
      passed += (before + after) * kStepWaves;
      wait_count(&sh.done, passed);
      kernel.fetch(then, sh.slot[turn ^ 1], 1);
    } else {
      wait_count(&sh.landed, rounds * kLoaders);
      switch (now.phase) {
        case kQkv: kernel.template run_product<kQkv>(now.layer, now.index, slot); break;
        case kAttend: kernel.run_attention(now.layer, now.index, slot); break;
        case kProj: kernel.template run_product<kProj>(now.layer, now.index, slot); break;
        case kUp: kernel.template run_product<kUp>(now.layer, now.index, slot); break;
        case kDown: kernel.template run_product<kDown>(now.layer, now.index, slot); break;
        case kPhases: kernel.run_last(now.index); break;
        default: break;
      }
      kernel.barrier();  // (the next task reuses the LDS)
    }
    task = next, now = then;
  }
}

// Clears the control words and marks all others as missing.  Bound by the launch.
constexpr int kFillThreads = 256;
__global__ __launch_bounds__(kFillThreads) void step_stack_fill_kernel(char *workspace, int64_t pieces) {
  for (int64_t i = (int64_t)blockIdx.x * kFillThreads + threadIdx.x; i < pieces; i += (int64_t)gridDim.x * kFillThreads) {
    const uint32_t w = i < kControlWords / 4 ? 0u : kMissing;
    store16(workspace + i * 16, Vec16{{w, w, w, w}});
  }
}

struct StackPlan {
  int64_t at_att, at_mid, at_act, at_h, at_part, layer_bytes;
  int steps, proj_splits, down_splits;
};

StackPlan stack_plan(const ic_step_stack_call &a) {
  const int es = elem_size(a.dtype);
  const int64_t q_cols = (int64_t)a.hn * a.hd, kv_cols = (int64_t)a.gn * a.hd;
  StackPlan s;
  // Steps of a wave in a task: a row of d in one task, since its norm needs all of it.
  s.steps = es == 2 ? 4 : a.d * es <= 6 * 64 * kStepWaves ? 6 : 8;
  auto splits = [&](int64_t k) { return (int)((k * es / 64 + s.steps * kStepWaves - 1) / (s.steps * kStepWaves)); };
  s.proj_splits = splits(q_cols), s.down_splits = splits(a.f);
  int64_t at = 0;
  auto take = [&](int64_t bytes) {
    const int64_t from = at;
    at += (bytes + 255) / 256 * 256;
    return from;
  };
  take(a.m * (q_cols + 2 * kv_cols) * es);
  s.at_att = take(a.m * q_cols * es);
  s.at_mid = take((int64_t)a.m * a.d * es);
  s.at_act = take((int64_t)a.m * a.f * es);
  s.at_h = take((int64_t)a.m * a.d * es);
  s.at_part = take((int64_t)(s.proj_splits - 1 + s.down_splits - 1) * a.m * a.d * 4);
  s.layer_bytes = at;
  return s;
}

template <class M, int HD, int GT, int S>
void launch_stack(const StackKP &kp, int workgroups, hipStream_t stream) {
  hipLaunchKernelGGL((step_stack_kernel<M, HD, GT, S>), dim3(workgroups), dim3(kStackThreads), 0, stream, kp);
}
template <class M, int HD, int GT>
void launch_steps(const StackKP &kp, int steps, int workgroups, hipStream_t stream) {
  if constexpr (sizeof(typename M::E::type) == 2)
    launch_stack<M, HD, GT, 4>(kp, workgroups, stream);
  else
    steps <= 6 ? launch_stack<M, HD, GT, 6>(kp, workgroups, stream) : launch_stack<M, HD, GT, 8>(kp, workgroups, stream);
}
template <class M, int HD>
void launch_group(const StackKP &kp, int steps, int workgroups, hipStream_t stream) {
  kp.dec.group == 1 ? launch_steps<M, HD, 1>(kp, steps, workgroups, stream) : launch_steps<M, HD, 4>(kp, steps, workgroups, stream);
}
template <class M>
void launch_typed(const StackKP &kp, int steps, int workgroups, hipStream_t stream) {
  kp.hd == 64 ? launch_group<M, 64>(kp, steps, workgroups, stream) : launch_group<M, 128>(kp, steps, workgroups, stream);
}

}  // namespace

size_t step_stack_workspace_bytes(const ic_step_stack_call &a) {
  return kControlWords * 4 + (size_t)a.num_layers * stack_plan(a).layer_bytes;
}

int launch_step_stack(const ic_step_stack_call &a, hipStream_t stream) {
  const StackPlan s = stack_plan(a);
  const int es = elem_size(a.dtype), tn = 64 / es;
  StackKP kp = {};
  for (int i = 0; i < a.num_layers; ++i) kp.layer[i] = a.layers[i];
  kp.x = (const char *)a.x, kp.out = (char *)a.out, kp.norm_out = (char *)a.norm_out;
  kp.last_weight = (const char *)a.norm_weight, kp.last_bias = (const char *)a.norm_bias;
  kp.last_norm = a.norm, kp.last_eps = a.eps;
  kp.control = (uint32_t *)a.workspace, kp.shared = (char *)a.workspace + kControlWords * 4;
  kp.layer_bytes = s.layer_bytes;
  kp.at_att = s.at_att, kp.at_mid = s.at_mid, kp.at_act = s.at_act, kp.at_h = s.at_h, kp.at_part = s.at_part;
  kp.layers = a.num_layers, kp.m = a.m, kp.d = a.d, kp.f = a.f;
  kp.act = a.act, kp.gated = a.act >= IC_ACT_GLU;
  kp.n_up = kp.gated ? 2 * a.f : a.f;
  kp.q_cols = a.hn * a.hd, kp.kv_cols = a.gn * a.hd;
  kp.tiles_d = (a.d + tn - 1) / tn, kp.proj_splits = s.proj_splits, kp.down_splits = s.down_splits;
  const int up = kp.gated ? tn / 2 : tn;
  const int tasks[kPhases] = {(kp.q_cols + tn - 1) / tn + (2 * kp.kv_cols + tn - 1) / tn, a.m * a.gn,
                              kp.tiles_d * s.proj_splits, (a.f + up - 1) / up, kp.tiles_d * s.down_splits};
  kp.first[0] = 0;
  for (int i = 0; i < kPhases; ++i) kp.first[i + 1] = kp.first[i] + tasks[i];
  kp.total = a.num_layers * kp.first[kPhases] + a.m;
  DecodeKP &dec = kp.dec;
  dec.block_tables = a.block_tables, dec.bt_stride = a.block_table_stride, dec.context_lens = a.context_lens;
  dec.stride_block = a.pool_stride_block, dec.stride_head = a.pool_stride_head, dec.stride_token = a.pool_stride_token;
  dec.num_blocks = a.num_blocks, dec.n_seqs = a.m, dec.hn = a.hn, dec.group = a.hn / a.gn;
  dec.max_ctx = a.max_context_len, dec.tiles_per_block = a.block_size / 16;
  dec.scale_log2e = a.scale * 1.4426950408889634f;
  kp.slots = a.slot_mapping, kp.positions = a.positions;
  kp.cos_table = a.cos_table, kp.sin_table = a.sin_table, kp.table_rows = a.table_rows;
  kp.num_slots = a.num_blocks * a.block_size;
  kp.gn = a.gn, kp.hd = a.hd, kp.must_draw = a.draw;
  kp.max_polls = (uint32_t)(a.max_polls > 0 ? a.max_polls : kMaxPolls), kp.status = a.status;
  kp.poll_mask = kp.max_polls < 1024 ? 0 : 1023;
  const int64_t pieces = (int64_t)step_stack_workspace_bytes(a) / 16;
  const int64_t fill = (pieces + kFillThreads - 1) / kFillThreads, most = 4 * (int64_t)device_cu_count();
  hipLaunchKernelGGL(step_stack_fill_kernel, dim3((unsigned)(fill < most ? fill : most)), dim3(kFillThreads), 0, stream,
                     (char *)a.workspace, pieces);
  const int workgroups = a.workgroups > 0 ? a.workgroups : device_cu_count();
  switch (a.dtype) {
    case IC_DTYPE_BF16: launch_typed<StepBf16>(kp, s.steps, workgroups, stream); break;
    case IC_DTYPE_F16: launch_typed<StepF16>(kp, s.steps, workgroups, stream); break;
    case IC_DTYPE_F32: launch_typed<StepF32>(kp, s.steps, workgroups, stream); break;
    default: return IC_ERR_UNSUPPORTED;
  }
  return hipGetLastError() == hipSuccess ? IC_OK : IC_ERR_LAUNCH;
}

}  // namespace ic
