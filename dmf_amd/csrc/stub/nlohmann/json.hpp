// torch's functorch headers name this third-party type in two inline members that serialise an interpreter; torch does not
// ship its header.  No data member has the type and nothing here calls those members, so declarations are all they need.
#pragma once
#include <string>

namespace nlohmann {
struct json {
  json() = default;
  template <typename T>
  explicit json(const T&);
  static json parse(const std::string&);
  template <typename T>
  T get() const;
  template <typename T>
  operator T() const;
  std::string dump() const;
};
}  // namespace nlohmann
