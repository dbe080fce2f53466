// A C entry must not let a C++ exception out: the SAH build, called while every
// allocation that librk.so itself makes on the C++ heap fails, still succeeds.
//
//   no_heap
// prints "status S", or "exception" (exit code 1).
#include <dlfcn.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <new>

#include "../../include/rk.h"
#include "../../include/rk_scenes.h"

static bool g_armed = false;

// Replaces the library's operator new too. The HIP runtime's calls go through.
void* operator new(size_t bytes) {
  Dl_info at;
  if (g_armed && dladdr(__builtin_return_address(0), &at) && at.dli_fname && std::strstr(at.dli_fname, "librk.so"))
    throw std::bad_alloc();
  void* p = std::malloc(bytes ? bytes : 1);
  if (!p) throw std::bad_alloc();
  return p;
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

template <typename T>
static T* device(size_t count, const T* from = nullptr) {
  void* p = nullptr;
  if (rk_malloc(&p, count * sizeof(T)) != RK_SUCCESS) std::exit(2);
  if (from && rk_memcpy(p, from, count * sizeof(T), 0, nullptr) != RK_SUCCESS) std::exit(2);
  return static_cast<T*>(p);
}

int main() {
  static rk_float4 verts[642];
  static rk_uint4 faces[1280];
  uint32_t nv = 0, n = 0;
  rk_aabox hitbox;
  if (rk_scene_icosphere(3, nullptr, nullptr, &nv, &n) != RK_SUCCESS || nv != 642 || n != 1280) return 2;
  if (rk_scene_icosphere(3, verts, faces, &nv, &n) != RK_SUCCESS) return 2;
  if (rk_scene_hitbox(verts, nv, &hitbox) != RK_SUCCESS) return 2;
  rk_uint4* f = device(n, faces);
  rk_float4* v = device(nv, verts);
  rk_aabox* boxes = device<rk_aabox>(n);
  uint32_t* ids = device<uint32_t>(n);
  rk_bvnode* nodes = device<rk_bvnode>(2 * n);
  uint32_t* info = device<uint32_t>(RK_INFO_WORDS);
  const size_t ws_bytes = rk_build_sah_workspace_size(n, 0);
  char* ws = device<char>(ws_bytes);
  try {
    g_armed = true;
    const rk_status s =
        rk_build_sah(nullptr, f, v, n, &hitbox, boxes, ids, nodes, 0, 2 * n, info, ws, ws_bytes);
    g_armed = false;
    std::printf("status %d\n", s);
    return s == RK_SUCCESS ? 0 : 1;
  } catch (const std::bad_alloc&) {
    g_armed = false;
    std::printf("exception\n");
    return 1;
  }
}
