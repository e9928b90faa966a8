import json,sys
a,b=[json.load(open(f)) for f in sys.argv[1:3]]
for k in a: print(f"{b[k]/a[k]:.3f} {a[k]:8.1f} {b[k]:8.1f} {k}{'   <<' if b[k]>1.02*a[k] else ''}")
