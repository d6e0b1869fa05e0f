// The analyses of a plan (direct.py, dkv_groups.py) and the padding of its block tables (executor.py), natively.
//
// What bounds preparing a plan is the host: a block is a Python object, the analyses look at each of some thousands two or
// three times, at 50-100 ns a look.  DCP plans every batch anew, so a training iteration pays for it.  Here a block is a
// few integers.  Backward plan of 16384 tokens, 16 heads, blocks of 512: the copies' analysis 494 -> 102 us, the
// replicas' 500 -> 110, the iteration 3.95 -> 2.44 ms; an iteration of 13.9 ms 6.5.  A plan off the wire has a string
// object a block, each told by its characters: 499 -> 259 and 504 -> 222.
//
// These functions take the plans that planners make: lists and tuples of BufferBlock, ReductionOp and SumOp
// themselves, plain integers and strings, slot numbers that index an array.  For anything else they return None and
// change nothing, and the Python code, which takes every plan, does it.
//
// They read a plan without owning it: its lists' storage, its blocks, its strings.  So nothing of Python's may run before
// the last look at it -- no call of a class or of an object's methods, and no new object that the garbage collector
// counts, since a collection runs finalisers and either may let another thread in, which may change the plan.  An analysis
// therefore has two parts: it reads the whole plan, and takes references to what the results hold; then it makes them.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <algorithm>
#include <cstdint>
#include <memory>
#include <new>
#include <utility>
#include <vector>

namespace {

struct NotTaken {};      // the plan has something that the Python code has to look at
struct PythonError {};   // a Python exception is set

// ---- Python objects ---------------------------------------------------------------------------------
struct Drop {
  void operator()(PyObject* o) const { Py_DECREF(o); }
};
typedef std::unique_ptr<PyObject, Drop> Ref;
Ref own(PyObject* o) {
  if (o == nullptr) throw PythonError();
  return Ref(o);
}
Ref share(PyObject* borrowed) {
  Py_INCREF(borrowed);
  return Ref(borrowed);
}
void check(int status) {
  if (status != 0) throw PythonError();
}

PyTypeObject *block_type, *reduction_op_type, *sum_op_type;  // set once by use_types
PyObject *s_buffer_type, *s_index, *s_n_tokens, *s_src_buffers, *s_dst_buffer;

PyObject* field(PyObject* o, PyObject* name) {  // of an instance of one of the classes above; borrowed
  PyObject** dict = _PyObject_GetDictPtr(o);
  if (dict == nullptr || *dict == nullptr) throw NotTaken();
  PyObject* value = PyDict_GetItemWithError(*dict, name);
  if (value == nullptr) {
    if (PyErr_Occurred()) throw PythonError();
    throw NotTaken();
  }
  return value;
}
struct Seq {  // a list or a tuple
  PyObject** items;
  Py_ssize_t n;
  explicit Seq(PyObject* o) {
    if (!PyList_CheckExact(o) && !PyTuple_CheckExact(o)) throw NotTaken();
    items = PySequence_Fast_ITEMS(o);
    n = PySequence_Fast_GET_SIZE(o);
  }
  PyObject* operator[](Py_ssize_t i) const { return items[i]; }
};
int64_t integer(PyObject* o) {
  if (!PyLong_CheckExact(o)) throw NotTaken();
  int overflow = 0;
  const long long v = PyLong_AsLongLongAndOverflow(o, &overflow);
  if (overflow != 0) throw NotTaken();
  return v;
}
constexpr int64_t kMaxIndex = (int64_t)1 << 22;  // of a slot: tables are arrays over them

// ---- blocks -----------------------------------------------------------------------------------------
enum : int { kLocalQ, kLocalKV, kLocaldQ, kLocaldKV, kLocalOut, kLocaldOut, kLocalLSE, kBufferQ, kBufferKV, kBufferdQ,
             kBufferdKV, kBufferOut, kBufferdOut, kBufferLSE, kKnownTypes };
const char* const kTypeNames[kKnownTypes] = {"LocalQ", "LocalKV", "LocaldQ", "LocaldKV", "LocalOut", "LocaldOut", "LocalLSE",
                                             "BufferQ", "BufferKV", "BufferdQ", "BufferdKV", "BufferOut", "BufferdOut", "BufferLSE"};
bool is_local(int type) { return type <= kLocalLSE; }
int local_of(int type) {  // what a slot of the type holds a copy of, if it is one
  switch (type) {
    case kBufferQ: return kLocalQ;
    case kBufferKV: return kLocalKV;
    case kBufferOut: return kLocalOut;
    case kBufferLSE: return kLocalLSE;
    case kBufferdOut: return kLocaldOut;
    default: return -1;
  }
}

struct Block {
  int type;
  int64_t index, n_tokens;
};

class Reader {
 public:
  Block block(PyObject* o) {
    const Block b = {type_of(o), slot(o), integer(field(o, s_n_tokens))};
    return b;
  }
  // parts of it, where the rest is not asked for: each is a look at memory that is in no cache
  int type_of(PyObject* o) {
    if (Py_TYPE(o) != block_type) throw NotTaken();
    return type(field(o, s_buffer_type));
  }
  static int64_t slot(PyObject* o) {
    if (Py_TYPE(o) != block_type) throw NotTaken();
    const int64_t index = integer(field(o, s_index));
    if (index < 0 || index >= kMaxIndex) throw NotTaken();
    return index;
  }

 private:
  // strings of a plan from a planner are the same few objects; one from the wire has an object of its own a block
  int type(PyObject* s) {
    for (const auto& [known, id] : seen_)
      if (known == s) return id;
    if (!PyUnicode_CheckExact(s)) throw NotTaken();
    for (int id = 0; id < kKnownTypes; ++id)
      if (PyUnicode_CompareWithASCIIString(s, kTypeNames[id]) == 0) {
        if (seen_.size() < 16) seen_.emplace_back(s, id);  // (the plan keeps it alive)
        return id;
      }
    throw NotTaken();
  }
  std::vector<std::pair<PyObject*, int>> seen_;
};

template <typename T>
class SlotMap {  // slot number -> T
 public:
  explicit SlotMap(T none) : none_(none) {}
  T get(int64_t i) const { return i < (int64_t)values_.size() ? values_[i] : none_; }
  void set(int64_t i, T v) {
    if (i >= (int64_t)values_.size()) values_.resize(std::max<size_t>(2 * values_.size(), i + 64), none_);
    values_[i] = v;
  }
  void drop(int64_t i) {
    if (i < (int64_t)values_.size()) values_[i] = none_;
  }

 private:
  T none_;
  std::vector<T> values_;
};

// ---- instructions -----------------------------------------------------------------------------------
// kinds[i] of the instructions, given by the caller (the exact class of each)
enum : int { kMemcpy = 0, kCommLaunch = 1, kBarrier = 2, kCommWait = 3, kAttn = 4, kAttnBackward = 5, kReduction = 6, kSum = 7 };

struct Instrs {
  Seq list;
  std::vector<int> kinds;
  std::vector<Ref> held;  // tables that are looked at
  Instrs(PyObject* instrs, PyObject* kind_list) : list(instrs) {
    const Seq k(kind_list);
    if (k.n != list.n) throw NotTaken();
    for (Py_ssize_t i = 0; i < k.n; ++i) kinds.push_back((int)integer(k[i]));
  }
  Py_ssize_t size() const { return list.n; }
  Seq table(Py_ssize_t i, const char* name) {
    held.push_back(own(PyObject_GetAttrString(list[i], name)));
    return Seq(held.back().get());
  }
  bool flag(Py_ssize_t i, const char* name) {
    const Ref value = own(PyObject_GetAttrString(list[i], name));
    if (PyBool_Check(value.get())) return value.get() == Py_True;
    return integer(value.get()) != 0;  // (any other object's truth is its own code's to say)
  }
};
Seq op_sources(PyObject* op, PyTypeObject* type) {
  if (Py_TYPE(op) != type) throw NotTaken();
  return Seq(field(op, s_src_buffers));
}
Seq pair_of(PyObject* o) {
  const Seq s(o);
  if (s.n != 2) throw NotTaken();
  return s;
}

// ---- which copies need not be made (direct.py: analyse) ---------------------------------------------
PyObject* direct(PyObject* instr_list, PyObject* kind_list) {
  Instrs instrs(instr_list, kind_list);
  Reader reader;
  struct Copy {  // of a local block
    int instr, pos;
    int64_t index, n_tokens;
  };
  std::vector<Copy> copies;
  std::vector<SlotMap<int>> origin(kKnownTypes, SlotMap<int>(-1));    // type -> slot -> its copy
  std::vector<SlotMap<int>> produced(kKnownTypes, SlotMap<int>(-1));  // type -> slot -> its producer
  struct Producer {
    int n_readers = 0, instr = 0, pos = 0;  // the last one
    bool scatter = false;                   // one source, unpadded
  };
  std::vector<Producer> producers;
  std::vector<std::vector<char>> copied(instrs.size());  // memcpy -> pair -> is it such a copy
  std::vector<int> first_producer(instrs.size(), 0);     // of an attention's rows or a sum's ops, in order
  struct Operands {
    bool has[4] = {false, false, false, false};  // q, kv, out, dq
    std::vector<int64_t> of[4];
    std::vector<int> kv_lengths;
  };
  std::vector<Operands> operands(instrs.size());
  std::vector<int> blocked;  // copies with a reader in their slot

  auto read_in_slot = [&](const Block& b) {
    const int c = origin[b.type].get(b.index);
    if (c >= 0) blocked.push_back(c);
  };
  auto overwritten = [&](int type, int64_t index) {
    origin[type].drop(index);
    produced[type].drop(index);
  };
  auto produce = [&](int type, int64_t index) {
    produced[type].set(index, (int)producers.size());
    producers.emplace_back();
  };
  auto read_by = [&](const Block& b, int instr, int pos, bool scatter) {
    const int who = produced[b.type].get(b.index);
    if (who < 0) return;
    Producer& p = producers[who];
    ++p.n_readers;
    p.instr = instr;
    p.pos = pos;
    p.scatter = scatter;
  };
  // the rows' blocks as indices of local blocks, where every one of them is a copy of one
  auto local_rows = [&](int type, const Seq& table, bool first_only, std::vector<int64_t>& to, std::vector<int>* lengths) -> bool {
    std::vector<Block> blocks;
    bool all = true;
    for (Py_ssize_t r = 0; r < table.n; ++r) {
      const Seq row(table[r]);
      if (first_only && row.n == 0) throw NotTaken();
      const Py_ssize_t n = first_only ? 1 : row.n;
      for (Py_ssize_t i = 0; i < n; ++i) {
        const Block b = reader.block(row[i]);
        blocks.push_back(b);
        const int c = b.type == type ? origin[type].get(b.index) : -1;
        if (c < 0 || copies[c].n_tokens != b.n_tokens) all = false;
        else to.push_back(copies[c].index);
      }
      if (lengths != nullptr) lengths->push_back((int)n);
    }
    if (!all)
      for (const Block& b : blocks) read_in_slot(b);
    return all;
  };
  auto first_of = [&](PyObject* row) {
    const Seq s(row);
    if (s.n == 0) throw NotTaken();
    return reader.block(s[0]);
  };

  for (Py_ssize_t idx = 0; idx < instrs.size(); ++idx) {
    const int kind = instrs.kinds[idx];
    if (kind == kMemcpy) {
      const Seq pairs = instrs.table(idx, "src_dst_pairs");
      copied[idx].assign(pairs.n, 0);
      for (Py_ssize_t pos = 0; pos < pairs.n; ++pos) {
        const Seq pair = pair_of(pairs[pos]);
        const Block src = reader.block(pair[0]);
        const int type = reader.type_of(pair[1]);
        const int64_t index = Reader::slot(pair[1]);
        produced[type].drop(index);
        if (src.type == local_of(type)) {
          origin[type].set(index, (int)copies.size());
          copies.push_back({(int)idx, (int)pos, src.index, src.n_tokens});
          copied[idx][pos] = 1;
        } else {
          origin[type].drop(index);
        }
      }
    } else if (kind == kAttn || kind == kAttnBackward) {
      Operands& mine = operands[idx];
      mine.has[0] = local_rows(kBufferQ, instrs.table(idx, "q_block_table"), true, mine.of[0], nullptr);
      mine.has[1] = local_rows(kBufferKV, instrs.table(idx, "kv_block_table"), false, mine.of[1], &mine.kv_lengths);
      const Seq out = instrs.table(idx, "out_block_table");
      if (kind == kAttn) {
        first_producer[idx] = (int)producers.size();
        for (Py_ssize_t b = 0; b < out.n; ++b) {
          const Block block = first_of(out[b]);
          overwritten(kBufferOut, block.index);
          overwritten(kBufferLSE, block.index);
          produce(kBufferOut, block.index);
        }
        continue;
      }
      // out, lse and dout of a row share the slot number: all three must be copies of the same local block
      const int types[3] = {kBufferOut, kBufferLSE, kBufferdOut};
      std::vector<int64_t> local[3];
      std::vector<int> hits;
      bool same = true;
      for (Py_ssize_t b = 0; b < out.n; ++b) {
        const Block block = first_of(out[b]);
        for (int t = 0; t < 3; ++t) {
          const int c = origin[types[t]].get(block.index);
          if (c >= 0) hits.push_back(c);
          if (c < 0 || copies[c].n_tokens != block.n_tokens) same = false;
          else local[t].push_back(copies[c].index);
        }
      }
      if (same && local[0] == local[1] && local[0] == local[2]) {
        mine.has[2] = true;
        mine.of[2] = std::move(local[0]);
      } else {
        blocked.insert(blocked.end(), hits.begin(), hits.end());
      }
      const Seq dq = instrs.table(idx, "dq_block_table"), dkv = instrs.table(idx, "dkv_block_table");
      first_producer[idx] = (int)producers.size();
      for (Py_ssize_t b = 0; b < dq.n; ++b) {
        const Block block = first_of(dq[b]);
        overwritten(block.type, block.index);
        produce(block.type, block.index);
      }
      for (Py_ssize_t b = 0; b < dkv.n; ++b) {
        const Seq row(dkv[b]);
        for (Py_ssize_t i = 0; i < row.n; ++i) overwritten(reader.type_of(row[i]), Reader::slot(row[i]));
      }
    } else if (kind == kReduction) {
      const Seq ops = instrs.table(idx, "ops");
      const bool unpadded = instrs.flag(idx, "output_is_unpadded");
      for (Py_ssize_t pos = 0; pos < ops.n; ++pos) {
        const Seq sources = op_sources(ops[pos], reduction_op_type);
        for (Py_ssize_t i = 0; i < sources.n; ++i) {
          const Seq pair = pair_of(sources[i]);
          const Block out = reader.block(pair[0]);
          read_in_slot(out);
          read_in_slot(reader.block(pair[1]));
          read_by(out, (int)idx, (int)pos, sources.n == 1 && unpadded);
        }
        if (unpadded) continue;
        const Seq dst = pair_of(field(ops[pos], s_dst_buffer));
        const Block out = reader.block(dst[0]), lse = reader.block(dst[1]);
        overwritten(out.type, out.index);
        overwritten(lse.type, lse.index);
        produce(out.type, out.index);
      }
    } else if (kind == kSum) {
      const Seq ops = instrs.table(idx, "ops");
      const bool unpadded = instrs.flag(idx, "output_is_unpadded");
      first_producer[idx] = (int)producers.size();
      for (Py_ssize_t pos = 0; pos < ops.n; ++pos) {
        const Seq sources = op_sources(ops[pos], sum_op_type);
        for (Py_ssize_t i = 0; i < sources.n; ++i) {
          const Block b = reader.block(sources[i]);
          read_by(b, (int)idx, (int)pos, sources.n == 1 && unpadded);
          read_in_slot(b);
        }
        if (unpadded) continue;
        const Block dst = reader.block(field(ops[pos], s_dst_buffer));
        overwritten(dst.type, dst.index);
        produce(dst.type, dst.index);
      }
    } else {
      throw NotTaken();
    }
  }

  // the op that scatters a result, where that is all that reads it
  auto sole_scatter = [&](int who) -> const Producer* {
    const Producer& p = producers[who];
    return p.n_readers == 1 && p.scatter ? &p : nullptr;
  };
  auto dst_of = [&](const Producer& p, int kind) {
    if (instrs.kinds[p.instr] != kind) throw NotTaken();
    const Seq ops = instrs.table(p.instr, "ops");
    return field(ops[p.pos], s_dst_buffer);
  };
  std::vector<std::pair<int, int>> skip_ops;
  struct Redirect {
    int instr, pos;
    Ref dst;
  };
  std::vector<Redirect> redirects;
  for (Py_ssize_t idx = 0; idx < instrs.size(); ++idx) {
    const int kind = instrs.kinds[idx];
    if (kind == kAttn || kind == kAttnBackward) {
      const Seq table = instrs.table(idx, kind == kAttn ? "out_block_table" : "dq_block_table");
      std::vector<const Producer*> hits;
      for (Py_ssize_t b = 0; b < table.n; ++b) {
        const Producer* p = sole_scatter(first_producer[idx] + (int)b);
        if (p == nullptr) break;
        hits.push_back(p);
      }
      if (table.n == 0 || (Py_ssize_t)hits.size() != table.n) continue;
      std::vector<int64_t> to;
      bool all = true;
      for (Py_ssize_t b = 0; b < table.n; ++b) {
        const Block mine = first_of(table[b]);
        PyObject* dst = dst_of(*hits[b], kind == kAttn ? kReduction : kSum);
        if (kind == kAttn) {
          const Seq pair = pair_of(dst);
          const Block out = reader.block(pair[0]), lse = reader.block(pair[1]);
          all &= out.type == kLocalOut && lse.type == kLocalLSE && out.n_tokens == mine.n_tokens;
          to.push_back(out.index);
        } else {
          const Block d = reader.block(dst);
          all &= d.type == kLocaldQ && d.n_tokens == mine.n_tokens;
          to.push_back(d.index);
        }
      }
      if (!all) continue;
      const int which = kind == kAttn ? 2 : 3;
      operands[idx].has[which] = true;
      operands[idx].of[which] = std::move(to);
      for (const Producer* p : hits) skip_ops.emplace_back(p->instr, p->pos);
    } else if (kind == kSum && !instrs.flag(idx, "output_is_unpadded")) {
      const Seq ops = instrs.table(idx, "ops");
      for (Py_ssize_t pos = 0; pos < ops.n; ++pos) {
        const Producer* p = sole_scatter(first_producer[idx] + (int)pos);
        if (p == nullptr) continue;
        PyObject* dst = dst_of(*p, kSum);
        const Block to = reader.block(dst);
        if (!is_local(to.type) || to.n_tokens != reader.block(field(ops[pos], s_dst_buffer)).n_tokens) continue;
        redirects.push_back({(int)idx, (int)pos, share(dst)});
        skip_ops.emplace_back(p->instr, p->pos);
      }
    }
  }
  for (const int c : blocked) copied[copies[c].instr][copies[c].pos] = 0;

  // ---- as Python objects (the plan is not looked at from here on) ----
  const Ref skip_pairs = own(PyDict_New()), operand_dict = own(PyDict_New()), skip_dict = own(PyDict_New()), redirect_dict = own(PyDict_New());
  auto entry = [](PyObject* dict, int64_t key, PyObject* (*make)()) {  // dict.setdefault(key, make()), borrowed
    const Ref k = own(PyLong_FromLongLong(key));
    PyObject* known = PyDict_GetItemWithError(dict, k.get());
    if (known != nullptr) return known;
    if (PyErr_Occurred()) throw PythonError();
    const Ref fresh = own(make());
    check(PyDict_SetItem(dict, k.get(), fresh.get()));
    return fresh.get();
  };
  auto new_set = +[]() { return PySet_New(nullptr); };
  auto new_dict = +[]() { return PyDict_New(); };
  auto add = [](PyObject* set, int64_t value) {
    const Ref v = own(PyLong_FromLongLong(value));
    check(PySet_Add(set, v.get()));
  };
  auto list_of = [](const int64_t* values, size_t n) {
    Ref list = own(PyList_New(n));
    for (size_t i = 0; i < n; ++i) PyList_SET_ITEM(list.get(), i, own(PyLong_FromLongLong(values[i])).release());
    return list;
  };
  for (Py_ssize_t idx = 0; idx < instrs.size(); ++idx) {
    for (size_t pos = 0; pos < copied[idx].size(); ++pos)
      if (copied[idx][pos]) add(entry(skip_pairs.get(), idx, new_set), pos);
    const char* const names[4] = {"q", "kv", "out", "dq"};
    for (int which = 0; which < 4; ++which) {
      const Operands& mine = operands[idx];
      if (!mine.has[which]) continue;
      Ref value;
      if (which == 1) {
        value = own(PyList_New(mine.kv_lengths.size()));
        size_t at = 0;
        for (size_t r = 0; r < mine.kv_lengths.size(); at += mine.kv_lengths[r], ++r)
          PyList_SET_ITEM(value.get(), r, list_of(mine.of[1].data() + at, mine.kv_lengths[r]).release());
      } else {
        value = list_of(mine.of[which].data(), mine.of[which].size());
      }
      check(PyDict_SetItemString(entry(operand_dict.get(), idx, new_dict), names[which], value.get()));
    }
  }
  for (const auto& [instr, pos] : skip_ops) add(entry(skip_dict.get(), instr, new_set), pos);
  for (const Redirect& r : redirects) {
    const Ref pos = own(PyLong_FromLong(r.pos));
    check(PyDict_SetItem(entry(redirect_dict.get(), r.instr, new_dict), pos.get(), r.dst.get()));
  }
  return PyTuple_Pack(4, skip_pairs.get(), operand_dict.get(), skip_dict.get(), redirect_dict.get());
}

// ---- which dK/dV replicas the backward kernel adds (dkv_groups.py: analyse, of launches not in parts) ----
std::vector<int> chunk_sizes(int n_visits, int limit) {
  std::vector<int> sizes(n_visits / limit - 1, limit);
  int left = n_visits - limit * (int)sizes.size();
  const int smallest = std::max(1, limit / 8);
  while (left > 0) {
    const int size = std::min(limit, std::max(smallest, (left + 1) / 2));
    sizes.push_back(std::min(size, left));
    left -= sizes.back();
  }
  return sizes;
}

PyObject* dkv(PyObject* instr_list, PyObject* kind_list, PyObject* limit_list, PyObject* redirect_ops, PyObject* group_type) {
  Instrs instrs(instr_list, kind_list);
  const Seq limits(limit_list);  // rows a group may visit, per instruction
  if (limits.n != instrs.size()) throw NotTaken();
  std::vector<SlotMap<PyObject*>> redirects(instrs.size(), SlotMap<PyObject*>(nullptr));  // sum -> position of an op -> where it goes
  {
    auto for_each = [](PyObject* dict, auto&& body) {  // (a lookup would compare its keys, with their own code)
      if (!PyDict_CheckExact(dict)) throw NotTaken();
      Py_ssize_t at = 0;
      PyObject *key, *value;
      while (PyDict_Next(dict, &at, &key, &value)) body(integer(key), value);
    };
    for_each(redirect_ops, [&](int64_t instr, PyObject* of_instr) {
      for_each(of_instr, [&](int64_t pos, PyObject* dst) {
        if (instr < 0 || instr >= instrs.size() || pos < 0 || pos >= kMaxIndex) throw NotTaken();
        redirects[instr].set(pos, dst);
      });
    });
  }
  Reader reader;
  constexpr int kUnread = -1, kElsewhere = -2;
  struct Visit {
    int row, pos;
    PyObject* slot;
    int64_t index, n_tokens;  // of the slot
    int reader;
  };
  std::vector<Visit> visits;
  std::vector<std::pair<int, int>> span(instrs.size(), {0, 0});  // a backward instruction's visits
  struct SumOf {
    int instr, pos;
    PyObject* op;
  };
  std::vector<SumOf> sums;
  SlotMap<int> written(-1), named(0);
  auto reads = [&](const Block& b, int who) {
    if (b.type == kBufferdKV) {
      const int v = written.get(b.index);
      if (v >= 0) visits[v].reader = visits[v].reader == kUnread ? who : kElsewhere;
    } else if (b.type == kLocaldKV) {
      named.set(b.index, named.get(b.index) + 1);
    }
  };
  auto writes = [&](const Block& b) {
    if (b.type == kBufferdKV) written.drop(b.index);
    else if (b.type == kLocaldKV) named.set(b.index, named.get(b.index) + 1);
  };
  for (Py_ssize_t idx = 0; idx < instrs.size(); ++idx) {
    const int kind = instrs.kinds[idx];
    if (kind == kAttnBackward) {
      const Seq table = instrs.table(idx, "dkv_block_table");
      span[idx].first = (int)visits.size();
      for (Py_ssize_t r = 0; r < table.n; ++r) {
        const Seq row(table[r]);
        for (Py_ssize_t i = 0; i < row.n; ++i) {
          const Block b = reader.block(row[i]);
          written.set(b.index, (int)visits.size());
          visits.push_back({(int)r, (int)i, row[i], b.index, b.n_tokens, kUnread});
        }
      }
      span[idx].second = (int)visits.size();
    } else if (kind == kSum) {
      const Seq ops = instrs.table(idx, "ops");
      for (Py_ssize_t pos = 0; pos < ops.n; ++pos) {
        const Seq sources = op_sources(ops[pos], sum_op_type);
        for (Py_ssize_t i = 0; i < sources.n; ++i) reads(reader.block(sources[i]), (int)sums.size());
        sums.push_back({(int)idx, (int)pos, ops[pos]});
      }
      for (Py_ssize_t pos = 0; pos < ops.n; ++pos) writes(reader.block(field(ops[pos], s_dst_buffer)));
    } else if (kind == kMemcpy) {
      const Seq pairs = instrs.table(idx, "src_dst_pairs");
      for (Py_ssize_t pos = 0; pos < pairs.n; ++pos) {
        const Seq pair = pair_of(pairs[pos]);
        const int from = reader.type_of(pair[0]), to = reader.type_of(pair[1]);
        if (from == kBufferdKV || from == kLocaldKV) reads(reader.block(pair[0]), kElsewhere);
        if (to == kBufferdKV || to == kLocaldKV) writes(reader.block(pair[1]));
      }
    } else if (kind == kReduction) {
      const Seq ops = instrs.table(idx, "ops");
      for (Py_ssize_t pos = 0; pos < ops.n; ++pos) {
        const Seq sources = op_sources(ops[pos], reduction_op_type);
        for (Py_ssize_t i = 0; i < sources.n; ++i) {
          const Seq pair = pair_of(sources[i]);
          for (int k = 0; k < 2; ++k) reads(reader.block(pair[k]), kElsewhere);
        }
        const Seq dst = pair_of(field(ops[pos], s_dst_buffer));
        for (int k = 0; k < 2; ++k) writes(reader.block(dst[k]));
      }
    } else if (kind != kAttn) {
      throw NotTaken();
    }
  }

  struct Group {
    std::vector<int> visits;
    PyObject* dst;  // borrowed from the plan while it is read
    int rank, component;
    Ref owned;  // dst
  };
  std::vector<std::pair<Py_ssize_t, std::vector<Group>>> groups_of;  // of the backward instructions
  std::vector<std::vector<char>> gone_of(sums.size());  // per sum op, its sources that the kernel has added already
  std::vector<char> filtered(sums.size(), 0), skipped(sums.size(), 0);
  // slot -> the latest of the ops below for which the kernel adds it (one map for all ops: it is as long as the highest
  // slot number, so that with one an op, 512 ops whose 66560 slots are the last below kMaxIndex took 168 ms, in Python
  // 131; now 80)
  SlotMap<int> added_for(0);
  int op_number = 0;
  for (Py_ssize_t idx = 0; idx < instrs.size(); ++idx) {
    if (instrs.kinds[idx] != kAttnBackward) continue;
    const int64_t limit64 = integer(limits[idx]);
    if (limit64 == 1) continue;
    if (limit64 < 1 || limit64 > 1024) throw NotTaken();
    const int limit = (int)limit64;
    // the rows' kv blocks, and the pairs' in the order of the visits
    const Seq table = instrs.table(idx, "kv_block_table");
    std::vector<std::vector<int64_t>> kv_rows(table.n);
    std::vector<int64_t> kv_of;
    for (Py_ssize_t r = 0; r < table.n; ++r) {
      const Seq row(table[r]);
      for (Py_ssize_t i = 0; i < row.n; ++i) kv_rows[r].push_back(Reader::slot(row[i]));
      kv_of.insert(kv_of.end(), kv_rows[r].begin(), kv_rows[r].end());
    }
    const int n = std::min<int>(span[idx].second - span[idx].first, (int)kv_of.size());
    // rows to take together: the same kv block, added by the same op and read by nothing else
    struct Together {
      int who;
      int64_t kv, n_tokens;
      std::vector<int> taken;
    };
    std::vector<Together> together;
    std::vector<int> alone;
    {
      SlotMap<int> last(-1);  // kv block -> the latest of `together` with it; the ones before it by `before`
      std::vector<int> before;
      for (int i = 0; i < n; ++i) {
        const int v = span[idx].first + i;
        const Visit& visit = visits[v];
        if (visit.reader < 0) {
          alone.push_back(v);
          continue;
        }
        int t = last.get(kv_of[i]);
        while (t >= 0 && (together[t].who != visit.reader || together[t].n_tokens != visit.n_tokens)) t = before[t];
        if (t < 0) {
          t = (int)together.size();
          together.push_back({visit.reader, kv_of[i], visit.n_tokens, {}});
          before.push_back(last.get(kv_of[i]));
          last.set(kv_of[i], t);
        }
        together[t].taken.push_back(v);
      }
    }
    // the order in which a group visits its rows: see _visit_order
    int number = 0;
    bool window = false;
    if (!together.empty() || !alone.empty()) {
      std::vector<std::pair<int, int>> counts;  // (number of rows, how many have it), in order of appearance
      auto count = [&](int rows, int times) {
        for (auto& c : counts)
          if (c.first == rows) {
            c.second += times;
            return;
          }
        counts.emplace_back(rows, times);
      };
      for (const Together& t : together) count((int)t.taken.size(), 1);
      if (!alone.empty()) count(1, (int)alone.size());
      std::pair<int, int> most = counts[0];
      for (const auto& c : counts)
        if (c.second > most.second) most = c;
      number = most.first;
      window = number > 2 && 2 * most.second > (int)(together.size() + alone.size());
    }
    std::vector<Group> groups;
    auto add_group = [&](std::vector<int> taken, PyObject* dst) { groups.push_back({std::move(taken), dst, 0, 0, nullptr}); };
    for (const int v : alone) add_group({v}, visits[v].slot);
    for (Together& t : together) {
      std::stable_sort(t.taken.begin(), t.taken.end(), [&](int a, int b) {
        const int ra = visits[a].row, rb = visits[b].row;
        if (window && ra % number != rb % number) return ra % number < rb % number;
        return ra > rb;
      });
      const SumOf& sum = sums[t.who];
      const Seq sources = op_sources(sum.op, sum_op_type);
      const int rows = (int)t.taken.size();
      PyObject* dst = redirects[sum.instr].get(sum.pos);  // where the sum goes, if that is an unpadded tensor
      if (dst == nullptr && instrs.flag(sum.instr, "output_is_unpadded")) dst = field(sum.op, s_dst_buffer);
      if (rows <= limit && rows == sources.n && dst != nullptr) {
        const Block to = reader.block(dst);
        if (to.type == kLocaldKV && to.n_tokens == visits[t.taken[0]].n_tokens && named.get(to.index) == 1) {
          add_group(t.taken, dst);
          skipped[t.who] = 1;
          continue;
        }
      }
      std::vector<char>& gone = gone_of[t.who];
      gone.resize(sources.n, 0);
      filtered[t.who] = 1;
      ++op_number;
      int at = 0;
      for (const int size : rows > limit ? chunk_sizes(rows, limit) : std::vector<int>{rows}) {
        add_group(std::vector<int>(t.taken.begin() + at, t.taken.begin() + at + size), visits[t.taken[at]].slot);
        for (int i = 1; i < size; ++i) added_for.set(visits[t.taken[at + i]].index, op_number);
        at += size;
      }
      for (Py_ssize_t i = 0; i < sources.n; ++i) {
        const Block b = reader.block(sources[i]);
        if (b.type == kBufferdKV && added_for.get(b.index) == op_number) gone[i] = 1;
      }
    }
    // kv blocks of one component: some row attends to both (see _components)
    SlotMap<int> node(-1);
    std::vector<int> parent;
    auto root = [&](int x) {
      while (parent[x] != x) x = parent[x] = parent[parent[x]];
      return x;
    };
    auto node_of = [&](int64_t kv) {
      int x = node.get(kv);
      if (x < 0) {
        x = (int)parent.size();
        parent.push_back(x);
        node.set(kv, x);
      }
      return x;
    };
    for (const auto& row : kv_rows) {
      if (row.empty()) continue;
      const int first = node_of(row[0]);
      for (const int64_t kv : row) {
        const int a = root(node_of(kv)), b = root(first);
        if (a != b) parent[std::max(a, b)] = std::min(a, b);
      }
    }
    std::vector<int> number_of(parent.size(), -1), members(parent.size(), 0), rank(parent.size()), component(parent.size());
    int n_components = 0;
    for (int x = 0; x < (int)parent.size(); ++x) {
      const int r = root(x);
      if (number_of[r] < 0) number_of[r] = n_components++;
      component[x] = number_of[r];
      rank[x] = members[r]++;
    }
    for (Group& g : groups) {
      const Visit& v = visits[g.visits[0]];
      if (v.row >= (int)kv_rows.size() || v.pos >= (int)kv_rows[v.row].size()) throw NotTaken();
      const int x = node.get(kv_rows[v.row][v.pos]);
      g.rank = rank[x];
      g.component = component[x];
    }
    std::stable_sort(groups.begin(), groups.end(), [](const Group& a, const Group& b) {
      if (a.visits.size() != b.visits.size()) return a.visits.size() > b.visits.size();
      return a.rank != b.rank ? a.rank < b.rank : a.component < b.component;
    });
    for (Group& g : groups) g.owned = share(g.dst);
    groups_of.emplace_back(idx, std::move(groups));
  }
  std::vector<std::vector<Ref>> left_of(sums.size());  // what a sum op still adds
  for (size_t who = 0; who < sums.size(); ++who) {
    if (!filtered[who]) continue;
    const Seq sources = op_sources(sums[who].op, sum_op_type);
    for (Py_ssize_t i = 0; i < sources.n; ++i)
      if (!gone_of[who][i]) left_of[who].push_back(share(sources[i]));
  }

  // ---- as Python objects (the plan is not looked at from here on) ----
  const Ref group_dict = own(PyDict_New()), skip_dict = own(PyDict_New()), source_dict = own(PyDict_New());
  for (const auto& [idx, groups] : groups_of) {
    const Ref list = own(PyList_New(groups.size()));
    for (size_t i = 0; i < groups.size(); ++i) {
      Ref pairs = own(PyList_New(groups[i].visits.size()));
      for (size_t k = 0; k < groups[i].visits.size(); ++k) {
        const Visit& v = visits[groups[i].visits[k]];
        Ref row = own(PyLong_FromLong(v.row)), pos = own(PyLong_FromLong(v.pos));
        PyList_SET_ITEM(pairs.get(), k, own(PyTuple_Pack(2, row.get(), pos.get())).release());
      }
      PyList_SET_ITEM(list.get(), i, own(PyObject_CallFunctionObjArgs(group_type, pairs.get(), groups[i].owned.get(), nullptr)).release());
    }
    const Ref key = own(PyLong_FromSsize_t(idx));
    check(PyDict_SetItem(group_dict.get(), key.get(), list.get()));
  }
  auto entry = [](PyObject* dict, int key, bool set) {
    const Ref k = own(PyLong_FromLong(key));
    PyObject* known = PyDict_GetItemWithError(dict, k.get());
    if (known != nullptr) return known;
    if (PyErr_Occurred()) throw PythonError();
    const Ref fresh = own(set ? PySet_New(nullptr) : PyDict_New());
    check(PyDict_SetItem(dict, k.get(), fresh.get()));
    return fresh.get();
  };
  for (size_t who = 0; who < sums.size(); ++who) {
    const Ref pos = own(PyLong_FromLong(sums[who].pos));
    if (skipped[who]) check(PySet_Add(entry(skip_dict.get(), sums[who].instr, true), pos.get()));
    if (!filtered[who]) continue;
    const Ref left = own(PyList_New(left_of[who].size()));
    for (size_t i = 0; i < left_of[who].size(); ++i) PyList_SET_ITEM(left.get(), i, left_of[who][i].release());
    check(PyDict_SetItem(entry(source_dict.get(), sums[who].instr, false), pos.get(), left.get()));
  }
  return PyTuple_Pack(3, group_dict.get(), skip_dict.get(), source_dict.get());
}

// ---- a block table as int32 [rows, width], filled up with -1 (executor.py: _padded) -------------------
// `rows`: of blocks (their slots), or of numbers that are looked up in `cu`; with `single`, a number a row.
bool padded(PyObject* row_list, Py_ssize_t width, PyObject* cu_list, bool single, int32_t* out, Py_ssize_t n_out) {
  const Seq rows(row_list);
  if (width < 1 || n_out / width != rows.n || n_out % width != 0) throw NotTaken();
  std::vector<int32_t> cu;
  if (cu_list != Py_None) {
    const Seq values(cu_list);
    for (Py_ssize_t i = 0; i < values.n; ++i) {
      const int64_t v = integer(values[i]);
      if (v < INT32_MIN || v > INT32_MAX) throw NotTaken();
      cu.push_back((int32_t)v);
    }
  }
  auto value = [&](PyObject* o) -> int32_t {
    int64_t v;
    if (cu_list == Py_None) {
      if (Py_TYPE(o) != block_type) throw NotTaken();
      v = integer(field(o, s_index));
      if (v < INT32_MIN || v > INT32_MAX) throw NotTaken();
      return (int32_t)v;
    }
    v = integer(o);
    if (v < 0 || v >= (int64_t)cu.size()) throw NotTaken();
    return cu[v];
  };
  for (Py_ssize_t r = 0; r < rows.n; ++r) {
    Py_ssize_t n = 1;
    if (single) {
      out[r * width] = value(rows[r]);
    } else {
      const Seq row(rows[r]);
      if (row.n > width) throw NotTaken();
      n = row.n;
      for (Py_ssize_t i = 0; i < n; ++i) out[r * width + i] = value(row[i]);
    }
    std::fill(out + r * width + n, out + (r + 1) * width, -1);
  }
  return true;
}

// ---- the module -------------------------------------------------------------------------------------
template <typename F>
PyObject* guarded(F&& body) {
  try {
    return body();
  } catch (const NotTaken&) {
    Py_RETURN_NONE;
  } catch (const PythonError&) {
    return nullptr;
  } catch (const std::bad_alloc&) {
    return PyErr_NoMemory();
  }
}

PyObject* py_use_types(PyObject*, PyObject* args) {
  PyObject *block, *reduction, *sum;
  if (!PyArg_ParseTuple(args, "O!O!O!", &PyType_Type, &block, &PyType_Type, &reduction, &PyType_Type, &sum)) return nullptr;
  for (PyObject* o : {block, reduction, sum}) Py_INCREF(o);  // (for as long as the process runs)
  block_type = (PyTypeObject*)block;
  reduction_op_type = (PyTypeObject*)reduction;
  sum_op_type = (PyTypeObject*)sum;
  Py_RETURN_NONE;
}
PyObject* py_direct(PyObject*, PyObject* args) {
  PyObject *instrs, *kinds;
  if (!PyArg_ParseTuple(args, "OO", &instrs, &kinds)) return nullptr;
  return guarded([&]() { return direct(instrs, kinds); });
}
PyObject* py_dkv(PyObject*, PyObject* args) {
  PyObject *instrs, *kinds, *limits, *redirects, *group;
  if (!PyArg_ParseTuple(args, "OOOOO", &instrs, &kinds, &limits, &redirects, &group)) return nullptr;
  return guarded([&]() { return dkv(instrs, kinds, limits, redirects, group); });
}
PyObject* py_padded(PyObject*, PyObject* args) {
  PyObject *rows, *cu;
  Py_ssize_t width;
  int single;
  Py_buffer out;
  if (!PyArg_ParseTuple(args, "OnOpw*", &rows, &width, &cu, &single, &out)) return nullptr;
  PyObject* result = guarded([&]() -> PyObject* {
    if (out.len % 4 != 0 || (reinterpret_cast<uintptr_t>(out.buf) & 3) != 0) throw NotTaken();
    return PyBool_FromLong(padded(rows, width, cu, single != 0, static_cast<int32_t*>(out.buf), out.len / 4));
  });
  PyBuffer_Release(&out);
  return result;
}

PyMethodDef methods[] = {
    {"use_types", py_use_types, METH_VARARGS, "the classes BufferBlock, ReductionOp and SumOp"},
    {"direct", py_direct, METH_VARARGS, "(skip_pairs, operands, skip_ops, redirect_ops) of DirectPlan, or None"},
    {"dkv", py_dkv, METH_VARARGS, "(groups, skip_ops, sources) of DkvGroups, or None"},
    {"padded", py_padded, METH_VARARGS, "fills an int32 table; None where it does not"},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_plan_analysis", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__plan_analysis(void) {
  s_buffer_type = PyUnicode_InternFromString("buffer_type");
  s_index = PyUnicode_InternFromString("index");
  s_n_tokens = PyUnicode_InternFromString("n_tokens");
  s_src_buffers = PyUnicode_InternFromString("src_buffers");
  s_dst_buffer = PyUnicode_InternFromString("dst_buffer");
  if (!s_buffer_type || !s_index || !s_n_tokens || !s_src_buffers || !s_dst_buffer) return nullptr;
  return PyModule_Create(&module);
}
