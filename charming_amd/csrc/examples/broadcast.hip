// Broadcasts (invoke_all) whose payload only thread 0 of the sender holds, to
// one chare a PE: every chare checks each payload's bytes.
//
//   word     chare 0 broadcasts `count` payloads of `bytes` from its thread
//            0's own memory; the other threads pass a null buffer.
//   full     the same while chare 1 keeps its PE busy for a bounded time with
//            most of its inbox taken, so that the broadcasts wait for room
//            there (or give up, with CHM_SPIN_LIMIT: ERR_SPIN_LIMIT).
//   self     more broadcasts than the sender's own inbox holds:
//            ERR_SELF_RING_FULL.
//
// argv: mode count bytes
#include <stdio.h>

#include <charming.h>

struct Node : charm::chare {
  int got, bad, done;
  __device__ Node() : got(0), bad(0), done(0) {}
  __device__ void start(void* arg);
  __device__ void take(void* arg);
  __device__ void report(void* arg);
  __device__ void hold(void* arg);
  __device__ void sink(void* arg);
};

__device__ void entry_start(Node& c, void* arg) { c.start(arg); }
__device__ void entry_take(Node& c, void* arg) { c.take(arg); }
__device__ void entry_report(Node& c, void* arg) { c.report(arg); }
__device__ void entry_hold(Node& c, void* arg) { c.hold(arg); }
__device__ void entry_sink(Node& c, void* arg) { c.sink(arg); }

constexpr int kMaxBytes = 64;
constexpr int kSinkBytes = 16000;

__shared__ charm::chare_proxy<Node>* node_proxy;
__device__ int g_mode, g_count, g_bytes;
__device__ char g_payload[kSinkBytes];

__device__ inline char expected(int k, int b) { return (char)(7 * k + 3 * b + 1); }

__device__ void charm::main(int argc, char** argv, size_t* argvs, int pe) {
  if (threadIdx.x == 0) {
    void* mem = charm::rt::heap_alloc(sizeof(charm::chare_proxy<Node>), 16);
    node_proxy = new (mem) charm::chare_proxy<Node>();
    node_proxy->add_entry_method<&entry_start>();
    node_proxy->add_entry_method<&entry_take>();
    node_proxy->add_entry_method<&entry_report>();
    node_proxy->add_entry_method<&entry_hold>();
    node_proxy->add_entry_method<&entry_sink>();
    node_proxy->create(charm::n_pes());
    if (pe == 0) {
      const char* m = argc > 1 ? argv[1] : "word";
      g_mode = (m[0] == 'f') ? 1 : (m[0] == 's') ? 2 : 0;
      g_count = argc > 2 ? charm::device_atoi(argv[2], argvs[2]) : 1;
      g_bytes = argc > 3 ? charm::device_atoi(argv[3], argvs[3]) : 4;
      if (g_bytes > kMaxBytes) g_bytes = kMaxBytes;
    }
  }
  __syncthreads();
  barrier();
  if (pe == 0) node_proxy->invoke(0, 0);
}

__device__ void Node::start(void* arg) {
  if (g_mode == 1) {
    node_proxy->invoke(1, 3);  // keep PE 1 busy first
    charm::flush_sends();
    for (int k = 0; k < 3; k++) node_proxy->invoke(1, 4, g_payload, kSinkBytes);
    charm::flush_sends();
  }
  alignas(16) char own[kMaxBytes];
  for (int k = 0; k < g_count; k++) {
    for (int b = 0; b < g_bytes; b++)
      own[b] = threadIdx.x == 0 ? expected(k, b) : (char)~expected(k, b);
    node_proxy->invoke_all(1, threadIdx.x == 0 ? own : nullptr, g_bytes);
  }
}

__device__ void Node::take(void* arg) {
  __shared__ int last;
  if (threadIdx.x == 0) {
    for (int b = 0; b < g_bytes; b++)
      if (((const char*)arg)[b] != expected(got, b)) {
        bad++;
        break;
      }
    last = ++got == g_count;
  }
  __syncthreads();
  if (last) node_proxy->invoke(0, 2, &bad, sizeof(int));
}

// chare 0: how many payloads each chare found wrong
__device__ void Node::report(void* arg) {
  __shared__ int all, wrong;
  if (threadIdx.x == 0) {
    if (done == 0) wrong = 0;
    wrong += *(const int*)arg;
    all = ++done == n;
    if (all)
      printf("Broadcast: %d payloads of %d bytes to %d chares, %d wrong\n",
             g_count, g_bytes, n, wrong);
  }
  __syncthreads();
  if (all) charm::end();
}

// occupy the PE for a bounded time, or until the runtime stops
__device__ void Node::hold(void* arg) {
  if (threadIdx.x == 0) {
    const double t0 = charm::wall_time();
    while (charm::wall_time() - t0 < 0.2 && !charm::rt::stopping())
      __builtin_amdgcn_s_sleep(8);
  }
  __syncthreads();
}

__device__ void Node::sink(void* arg) {}
