// Captures by name: what a captured call points at (block maps, id arrays) has to live as long as the graph that reads it, and no
// longer.  HIP tells when that is: a user object retained by a graph passes to the executables made of it and is destroyed with the
// last of them.  Host code only.
#include <mutex>
#include <unordered_map>
#include <vector>

#include "flexattn.h"
#include "launch.hpp"

namespace {

struct Captures {
  std::mutex mutex;
  std::unordered_map<unsigned long long, int64_t> tokens;   // HIP's id of a capture whose graph lives -> its token
  std::vector<int64_t> ended;                               // tokens of graphs that are gone, not yet fetched
  int64_t last = 0;
};
// (never destroyed: graphs may outlive this library's static objects)
Captures& captures() {
  static Captures* c = new Captures;
  return *c;
}

struct Note {
  unsigned long long id;
  int64_t token;
};
// (from whichever thread drops the graph: no HIP call and nothing that waits)
void graph_gone(void* p) {
  Note* note = static_cast<Note*>(p);
  Captures& c = captures();
  std::lock_guard<std::mutex> lock(c.mutex);
  const auto it = c.tokens.find(note->id);
  if (it != c.tokens.end() && it->second == note->token) c.tokens.erase(it);
  c.ended.push_back(note->token);
  delete note;
}

}  // namespace

using namespace fa;

extern "C" {

int64_t flexattn_capture_token(void* stream) {
  if (stream == nullptr) return 0;   // (the default stream is never captured)
  hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
  unsigned long long id = 0;
  hipGraph_t graph = nullptr;
  hipError_t e = hipStreamGetCaptureInfo_v2(static_cast<hipStream_t>(stream), &status, &id, &graph, nullptr, nullptr);
  if (e != hipSuccess) return set_error(FLEXATTN_ELAUNCH, "hipStreamGetCaptureInfo: %s", hipGetErrorString(e));
  if (status != hipStreamCaptureStatusActive || graph == nullptr) return 0;
  Captures& c = captures();
  Note* note = nullptr;
  {
    std::lock_guard<std::mutex> lock(c.mutex);
    const auto it = c.tokens.find(id);
    if (it != c.tokens.end()) return it->second;
    note = new Note{id, ++c.last};
    c.tokens[id] = note->token;
  }
  const int64_t token = note->token;
  hipUserObject_t object = nullptr;
  e = hipUserObjectCreate(&object, note, graph_gone, 1, hipUserObjectNoDestructorSync);
  if (e == hipSuccess) e = hipGraphRetainUserObject(graph, object, 1, hipGraphUserObjectMove);
  if (e != hipSuccess) (void)hipGetLastError();   // (a graph whose end nothing will tell: what it reads is kept)
  return token;
}

int32_t flexattn_captures_ended(int64_t* tokens, int32_t n) {
  if (tokens == nullptr || n <= 0) return 0;
  Captures& c = captures();
  std::lock_guard<std::mutex> lock(c.mutex);
  int32_t i = 0;
  for (; i < n && !c.ended.empty(); ++i) {
    tokens[i] = c.ended.back();
    c.ended.pop_back();
  }
  return i;
}

}  // extern "C"
